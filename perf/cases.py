"""What is timed of this framework: the int4 linear, its GPTQ module, prompt layers and the
captured decode steps, at the sizes of the Qwen3-8B-shaped MOSS-TTS backbone.

``listed()`` names the cases, ``draw(rng)`` gives others of the same ranges, ``prepare``
builds what a program holds before the call (weights, caches, a captured graph), ``run`` is
one pass through the public entry points, ``exact`` the same values from plain torch in
float64, ``work`` what a pass cannot do without and ``tolerance`` how far another correct
implementation may be from it.

Four kinds of case:

* ``op``: ``ops.weight_int4pack_mm`` on the reference's ``(packed, qsz)`` records;
* ``gptq``: the forward of a ``GPTQLinear`` (AutoGPTQ buffers, act-order or not);
* ``prompt``: ``prefill_rows`` of a one-layer backbone, the layer's output rows and the K/V
  rows it writes;
* ``step``: one replayed decode step at a position of a filled KV cache, its logits and the
  K/V rows of that position.
"""
from __future__ import annotations

import math

import torch

import __graft_entry__

__graft_entry__.import_package()

from moss_tts_lite_amd import fast, gptq, model, ops  # noqa: E402

HIDDEN, INTER, HEADS, KV_HEADS, DIM = 4096, 12288, 32, 8, 128
QKV, KV = (HEADS + 2 * KV_HEADS) * DIM, KV_HEADS * DIM
VOCAB, MOSS_VOCAB, N_VQ, AUDIO_VOCAB, PAD_CODE = 151936, 155648, 32, 1025, 1024
TWO_WAY = (151656, 151662)
SHORT_VOCAB = 4096            # rows of the embedding and head where a case is about the layers
THETA, EPS = 1_000_000.0, 1e-6


def listed() -> list[dict]:
    return [
        # the gate|up GEMV of every decode step, as the eager drop-in operator runs it
        {"name": "op_row_gate_up", "kind": "op", "m": 1, "k": 4096, "n": 24576, "g": 128},
        # a handful of rows (several candidates or a short continuation) through down
        {"name": "op_rows_down", "kind": "op", "m": 7, "k": 12288, "n": 4096, "g": 128},
        # a one-sentence prompt through the fused q|k of the shipped g32 preset
        {"name": "op_prompt_qk", "kind": "op", "m": 61, "k": 4096, "n": 5120, "g": 32},
        # a paragraph with a reference clip through gate|up of the same preset
        {"name": "op_prompt_gate_up", "kind": "op", "m": 389, "k": 4096, "n": 24576, "g": 32},
        # a long text with a long reference clip through down
        {"name": "op_prompt_down", "kind": "op", "m": 1536, "k": 12288, "n": 4096, "g": 128},
        # the smallest call: one row through an act-order o projection
        {"name": "gptq_row_o", "kind": "gptq", "m": 1, "k": 4096, "n": 4096, "g": 128,
         "act_order": True},
        # a prompt through the act-order gate|up module, outside the captured decoder
        {"name": "gptq_prompt_gate_up", "kind": "gptq", "m": 200, "k": 4096, "n": 24576,
         "g": 128, "act_order": True},
        # the benchmark's 256-token prompt, one of its act-order g128 layers
        {"name": "prompt_layer", "kind": "prompt", "rows": 256, "moss": False, "g": 128},
        # a voice-cloning prompt (text and a reference clip of a minute and a half), one
        # MOSS layer of the g32 preset with its bf16 v_proj
        {"name": "prompt_layer_moss", "kind": "prompt", "rows": 1100, "moss": True, "g": 32},
        # the benchmark's greedy step in the middle of its range
        {"name": "step", "kind": "step", "pos": 768, "layers": 36, "moss": False, "g": 128,
         "max_seq": 2048, "vocab": VOCAB, "audio2": False},
        # one audio frame of a MOSS generation two minutes in
        {"name": "step_moss", "kind": "step", "pos": 1500, "layers": 36, "moss": True, "g": 32,
         "max_seq": 4096, "vocab": MOSS_VOCAB, "audio2": True},
        # a step late in a long document, two layers (attention over a long cache)
        {"name": "step_long", "kind": "step", "pos": 6000, "layers": 2, "moss": False, "g": 128,
         "max_seq": 8192, "vocab": SHORT_VOCAB, "audio2": False},
    ]


_SHAPES = ((4096, 6144), (4096, 5120), (4096, 4096), (4096, 24576), (12288, 4096),
           (4096, 12288), (4096, 1024))


def _log(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(("op", "op", "op", "gptq", "gptq", "prompt", "prompt", "step"))
    g = rng.choice((32, 32, 64, 128, 128, 256))
    if kind in ("op", "gptq"):
        if rng.random() < 0.2:      # a model of another width
            k, n = 256 * rng.randint(2, 24), 16 * rng.randint(20, 600)
        else:
            k, n = rng.choice(_SHAPES)
        case = {"kind": kind, "m": _log(rng, 1, 1536 if kind == "op" else 600), "k": k, "n": n,
                "g": g}
        if kind == "gptq":
            case["act_order"] = rng.random() < 0.7
        return case
    if kind == "prompt":
        moss = rng.random() < 0.5
        return {"kind": kind, "rows": _log(rng, 12, 1100), "moss": moss,
                "g": rng.choice((32, 32, 128)) if moss else rng.choice((64, 128, 128))}
    if rng.random() < 0.5:          # the whole model
        moss = rng.random() < 0.5
        return {"kind": kind, "pos": _log(rng, 16, 2000), "layers": 36, "moss": moss,
                "g": 32 if moss else 128, "max_seq": 2048,
                "vocab": MOSS_VOCAB if moss else VOCAB, "audio2": moss and rng.random() < 0.7}
    return {"kind": kind, "pos": rng.randint(1500, 8100), "layers": 2, "moss": False,
            "g": rng.choice((64, 128)), "max_seq": 8192, "vocab": SHORT_VOCAB, "audio2": False}


# ------------------------------------------------------------------------------ inputs
def _gen(seed: int, stream: int = 0) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1009 + stream)
    return g


def _normal(gen, *shape, std=1.0) -> torch.Tensor:
    return torch.randn(*shape, device="cuda", generator=gen).mul_(std).bfloat16()


def _activations(gen, m: int, k: int) -> torch.Tensor:
    """Normed activations: unit scale, one channel in 256 eight times as large."""
    x = torch.randn(m, k, device="cuda", generator=gen)
    x[:, torch.randint(0, k, (k // 256,), device="cuda", generator=gen)] *= 8.0
    return x.bfloat16()


def _qsz_record(gen, n: int, k: int, g: int):
    """Pre-packed codes uint8 [N, K/2] (even k in the high nibble) and qsz bf16 [K/g, N, 2]."""
    pre = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device="cuda", generator=gen)
    s = torch.rand(k // g, n, device="cuda", generator=gen) * 0.004 + 0.002
    z = torch.randn(k // g, n, device="cuda", generator=gen) * 0.002
    return pre, torch.stack([s, z], -1).bfloat16()


def _qsz_weight(rec, g: int) -> torch.Tensor:
    """The record's weight in float64, [N, K]."""
    pre, qsz = rec
    q = torch.stack([pre >> 4, pre & 15], -1).reshape(pre.shape[0], -1)
    s, z = (qsz[..., i].t().double().repeat_interleave(g, 1) for i in (0, 1))
    return (q.double() - 8.0).mul_(s).add_(z)


def _gptq_buffers(gen, k: int, n: int, g: int, act_order: bool, g_idx=None):
    """qweight, zeros (uint8, unpacked), scales fp16 and g_idx of an AutoGPTQ linear."""
    qweight = torch.randint(-2**31, 2**31 - 1, (k // 8, n), dtype=torch.int32, device="cuda",
                            generator=gen)
    scales = (torch.rand(k // g, n, device="cuda", generator=gen) * 0.004 + 0.002).half()
    zeros = torch.randint(6, 10, (k // g, n), dtype=torch.uint8, device="cuda", generator=gen)
    if act_order:
        g_idx = torch.empty(k, dtype=torch.int32, device="cuda")
        g_idx[torch.randperm(k, device="cuda", generator=gen)] = (
            torch.arange(k, device="cuda") // g).int()
    return qweight, zeros, scales, g_idx


def _pack_zeros(zeros: torch.Tensor) -> torch.Tensor:
    z = zeros.to(torch.int64).reshape(zeros.shape[0], -1, 8)
    word = sum(z[..., j] << (4 * j) for j in range(8))
    return ((word + 2**31) % 2**32 - 2**31).to(torch.int32)


def _gptq_linear(buf, g: int) -> gptq.GPTQLinear:
    qweight, zeros, scales, g_idx = buf
    return gptq.GPTQLinear.from_buffers(qweight, _pack_zeros(zeros), scales, g_idx, g)


def _gptq_weight(buf, g: int) -> torch.Tensor:
    """The linear's weight in float64, [N, K]."""
    qweight, zeros, scales, g_idx = buf
    k, n = qweight.shape[0] * 8, qweight.shape[1]
    q = torch.stack([(qweight >> (4 * j)) & 15 for j in range(8)], 1).reshape(k, n)
    grp = (torch.arange(k, device="cuda") // g) if g_idx is None else g_idx.long()
    return (q.double() - zeros.double()[grp]).mul_(scales.double()[grp]).t()


_LINEARS = (("qkv", HIDDEN, QKV), ("o", HIDDEN, HIDDEN), ("gate_up", HIDDEN, 2 * INTER),
            ("down", INTER, HIDDEN))


def _layer_tensors(case: dict, seed: int, li: int) -> dict:
    """One layer's norms and linears.  The benchmark form holds four act-order GPTQ linears
    (gate|up in alternating 32-column blocks); the MOSS form the preset's records with v_proj
    in bf16."""
    gen = _gen(seed, 1 + li)
    out = {k: (1.0 + 0.05 * torch.randn(w, device="cuda", generator=gen)).bfloat16()
           for k, w in (("input_layernorm", HIDDEN), ("post_attention_layernorm", HIDDEN),
                        ("q_norm", DIM), ("k_norm", DIM))}
    if case["moss"]:
        for name, k, n in (("qk", HIDDEN, QKV - KV), ("o", HIDDEN, HIDDEN), ("gate", HIDDEN, INTER),
                           ("up", HIDDEN, INTER), ("down", INTER, HIDDEN)):
            out[name] = _qsz_record(gen, n, k, case["g"])
        out["v"] = _normal(gen, KV, HIDDEN, std=0.02)
    else:
        for name, k, n in _LINEARS:
            out[name] = _gptq_buffers(gen, k, n, case["g"], True)
    return out


def _layer_weights(case: dict, t: dict) -> dict:
    """The tensors as the backbone takes them."""
    g = case["g"]
    out = {k: t[k] for k in ("input_layernorm", "post_attention_layernorm", "q_norm", "k_norm")}
    if case["moss"]:
        lin = {k: gptq.QszLinear(ops.convert_weight_to_int4pack(t[k][0], 8), t[k][1], g)
               for k in ("qk", "o", "gate", "up", "down")}
        out.update(qkv=lin["qk"], o=lin["o"], down=lin["down"], v=t["v"],
                   gate_up=gptq.interleave_qsz_gate_up(lin["gate"], lin["up"]))
    else:
        out.update({name: _gptq_linear(t[name], g) for name, _, _ in _LINEARS})
    return out


def _layer_matrices(case: dict, t: dict) -> dict:
    """The layer's float64 weights [N, K]: qkv, o, gate, up, down."""
    g = case["g"]
    if case["moss"]:
        w = {k: _qsz_weight(t[k], g) for k in ("o", "gate", "up", "down")}
        w["qkv"] = torch.cat([_qsz_weight(t["qk"], g), t["v"].double()])
        return w
    w = {k: _gptq_weight(t[k], g) for k in ("qkv", "o", "down")}
    gu = _gptq_weight(t["gate_up"], g).reshape(INTER // 32, 2, 32, HIDDEN)
    w["gate"], w["up"] = gu[:, 0].reshape(INTER, HIDDEN), gu[:, 1].reshape(INTER, HIDDEN)
    return w


def _tables(case: dict, seed: int) -> dict:
    """Embeddings, final norm and heads."""
    gen = _gen(seed)
    vocab = case.get("vocab", SHORT_VOCAB)
    out = {"embed_tokens": _normal(gen, vocab, HIDDEN),
           "final_norm": (1.0 + 0.05 * torch.randn(HIDDEN, device="cuda", generator=gen)).bfloat16(),
           "head": _normal(gen, vocab, HIDDEN, std=0.02)}
    if case["moss"]:
        out["emb_ext"] = list(_normal(gen, N_VQ, AUDIO_VOCAB, HIDDEN, std=0.2))
        out["head_audio"] = _normal(gen, N_VQ, AUDIO_VOCAB, HIDDEN, std=0.02)
    return out


def _ids(case: dict, seed: int, rows: int) -> torch.Tensor:
    gen = _gen(seed, 1000)
    limit = case.get("vocab", SHORT_VOCAB)
    ids = torch.randint(0, limit, (rows, 1), device="cuda", generator=gen)
    if case["moss"]:
        audio = torch.randint(0, AUDIO_VOCAB, (rows, N_VQ), device="cuda", generator=gen)
        ids = torch.cat([ids, audio], 1)
    return ids


def _cache(case: dict, seed: int, li: int):
    """The K and V rows [kv_heads, pos, 128] that the positions before the step have left."""
    gen = _gen(seed, 2000 + li)
    return (_normal(gen, KV_HEADS, case["pos"], DIM), _normal(gen, KV_HEADS, case["pos"], DIM))


def _config(case: dict) -> model.BackboneConfig:
    vocab = case.get("vocab", SHORT_VOCAB)
    cfg = dict(hidden=HIDDEN, n_heads=HEADS, n_kv_heads=KV_HEADS, head_dim=DIM,
               intermediate=INTER, n_layers=case.get("layers", 1), vocab=vocab,
               group_size=case["g"], act_order=not case["moss"], rope_theta=THETA, eps=EPS,
               max_seq=case.get("max_seq", 2048))
    if case["moss"]:
        cfg.update(n_vq=N_VQ, audio_vocab=AUDIO_VOCAB, audio_pad_code=PAD_CODE,
                   two_way_ids=TWO_WAY if vocab > max(TWO_WAY) else (0, 1))
    return model.BackboneConfig(**cfg)


def _decoder(case: dict, seed: int):
    cfg = _config(case)
    weights = _tables(case, seed)
    weights["layers"] = [_layer_weights(case, _layer_tensors(case, seed, li))
                         for li in range(cfg.n_layers)]
    backbone = model.Int4Backbone(cfg, weights).keep_strip_copies_only()
    return (fast.FastMossDecoder if case["moss"] else fast.FastDecoder)(backbone)


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "op":
        gen = _gen(seed)
        pre, qsz = _qsz_record(gen, case["n"], case["k"], case["g"])
        return {"case": case, "x": _activations(gen, case["m"], case["k"]), "qsz": qsz,
                "packed": ops.convert_weight_to_int4pack(pre, 8)}
    if kind == "gptq":
        gen = _gen(seed)
        buf = _gptq_buffers(gen, case["k"], case["n"], case["g"], case["act_order"])
        return {"case": case, "x": _activations(gen, case["m"], case["k"]),
                "linear": _gptq_linear(buf, case["g"]).post_init()}
    dec = _decoder(case, seed)
    if kind == "prompt":
        return {"case": case, "dec": dec, "ids": _ids(case, seed, case["rows"])}
    for li in range(case["layers"]):
        k, v = _cache(case, seed, li)
        dec.m.k_cache[li, :, :case["pos"]] = k
        dec.m.v_cache[li, :, :case["pos"]] = v
    # the capture's warm-up steps write at the position the step then rewrites
    dec.pos.fill_(case["pos"])
    dec.capture()
    ids = _ids(case, seed, 1)[0]
    return {"case": case, "dec": dec, "row": ids, "token": int(ids[0])}


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "op":
        return ops.weight_int4pack_mm(state["x"], state["packed"], case["g"], state["qsz"])
    if kind == "gptq":
        return state["linear"](state["x"])
    dec = state["dec"]
    if kind == "prompt":
        rows = case["rows"]
        h = dec.prefill_rows(state["ids"])
        return {"h": h, "k": dec.m.k_cache[0, :, :rows], "v": dec.m.v_cache[0, :, :rows]}
    pos = case["pos"]
    kv = {"k": dec.m.k_cache[:, :, pos], "v": dec.m.v_cache[:, :, pos]}
    if not case["moss"]:
        dec.step(state["token"], pos)
        return {"logits": dec.logits, **kv}
    lt, la, h, two = dec.step(state["row"], pos, case["audio2"])
    return {"first": two if case["audio2"] else lt, "audio": la, "h": h, **kv}


# ------------------------------------------------------------------------- float64 values
def _norm64(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x: torch.Tensor, pos0: int) -> torch.Tensor:
    """Rotary embedding of x [rows, heads, 128] at pos0 .., from the bf16 tables the model
    holds (float32 angles)."""
    inv = 1.0 / (THETA ** (torch.arange(0, DIM, 2, dtype=torch.float32, device="cuda") / DIM))
    t = torch.arange(pos0 + x.shape[0], dtype=torch.float32, device="cuda")[pos0:]
    a = torch.outer(t, inv)
    a = torch.cat([a, a], -1)[:, None]
    half = torch.cat([-x[..., DIM // 2:], x[..., :DIM // 2]], -1)
    return x * a.cos().bfloat16().double() + half * a.sin().bfloat16().double()


def _layer64(case: dict, t: dict, h: torch.Tensor, pos0: int, past=None):
    """One decoder layer on h [rows, hidden] (float64): its output and K/V [kv_heads, rows, 128]."""
    w = _layer_matrices(case, t)
    rows = h.shape[0]
    y = _norm64(h, t["input_layernorm"]) @ w["qkv"].t()
    q, k, v = (s.reshape(rows, -1, DIM) for s in y.split([HEADS * DIM, KV, KV], -1))
    q = _rope64(_norm64(q, t["q_norm"]), pos0).transpose(0, 1)
    k = _rope64(_norm64(k, t["k_norm"]), pos0).transpose(0, 1)
    v = v.transpose(0, 1)
    keys, vals = (k, v) if past is None else (torch.cat([p.double(), n], 1)
                                              for p, n in zip(past, (k, v)))
    heads = []
    causal = torch.arange(keys.shape[1], device="cuda")[None] <= \
        pos0 + torch.arange(rows, device="cuda")[:, None]
    for i in range(HEADS):
        j = i // (HEADS // KV_HEADS)
        s = (q[i] @ keys[j].t() / math.sqrt(DIM)).masked_fill(~causal, float("-inf"))
        heads.append(torch.softmax(s, -1) @ vals[j])
    h = h + torch.cat(heads, -1) @ w["o"].t()
    x = _norm64(h, t["post_attention_layernorm"])
    act = torch.nn.functional.silu(x @ w["gate"].t()) * (x @ w["up"].t())
    return h + act @ w["down"].t(), k, v


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("op", "gptq"):
        gen = _gen(seed)
        if kind == "op":
            w = _qsz_weight(_qsz_record(gen, case["n"], case["k"], case["g"]), case["g"])
        else:
            w = _gptq_weight(_gptq_buffers(gen, case["k"], case["n"], case["g"],
                                           case["act_order"]), case["g"])
        return _activations(gen, case["m"], case["k"]).double() @ w.t()
    tab = _tables(case, seed)
    rows = case["rows"] if kind == "prompt" else 1
    ids = _ids(case, seed, rows)
    h = tab["embed_tokens"][ids[:, 0]].double()
    for i, emb in enumerate(tab.get("emb_ext", ())):
        h = h + emb[ids[:, 1 + i]].double()
    if kind == "prompt":
        h, k, v = _layer64(case, _layer_tensors(case, seed, 0), h, 0)
        return {"h": h, "k": k, "v": v}
    ks, vs = [], []
    for li in range(case["layers"]):
        h, k, v = _layer64(case, _layer_tensors(case, seed, li), h, case["pos"],
                           _cache(case, seed, li))
        ks.append(k[:, 0])
        vs.append(v[:, 0])
    kv = {"k": torch.stack(ks), "v": torch.stack(vs)}
    hf = _norm64(h, tab["final_norm"])[0]
    if not case["moss"]:
        return {"logits": tab["head"].double() @ hf, **kv}
    head = tab["head"][list(_config(case).two_way_ids)] if case["audio2"] else tab["head"]
    audio = tab["head_audio"].double() @ hf
    audio[:, PAD_CODE] = float("-inf")
    return {"first": head.double() @ hf, "audio": audio, "h": hf, **kv}


# --------------------------------------------------------------------------------- work
def _linear_bytes(k: int, n: int, g: int, moss: bool) -> float:
    """The weight and its group metadata, once."""
    return n * k / 2 + (k // g) * n * (4 if moss else 2.5)


def work(case: dict) -> dict:
    kind, g = case["kind"], case["g"]
    if kind in ("op", "gptq"):
        m, k, n = case["m"], case["k"], case["n"]
        nbytes = _linear_bytes(k, n, g, kind == "op") + 2 * m * (k + n)
        return {"bytes": nbytes + (4 * k if case.get("act_order") else 0), "flops": 2.0 * m * n * k}
    moss = case["moss"]
    rows = case["rows"] if kind == "prompt" else 1
    past = 0 if kind == "prompt" else case["pos"]
    layers = case.get("layers", 1)
    nbytes = _linear_bytes(HIDDEN, QKV - (KV if moss else 0), g, moss) + \
        (2 * KV * HIDDEN if moss else 0) + sum(_linear_bytes(k, n, g, moss)
                                               for _, k, n in _LINEARS[1:])
    nbytes += 4 * KV * (past + rows)                      # K and V read and written
    weights = sum(k * n for _, k, n in _LINEARS)
    pairs = rows * past + rows * (rows + 1) // 2          # (query, key) pairs of a head
    flops = 2.0 * rows * weights + 4.0 * HEADS * DIM * pairs
    total = {"bytes": layers * nbytes, "flops": layers * flops}
    total["bytes"] += 2 * HIDDEN * rows * (1 + (N_VQ if moss else 0) + 1)
    if kind == "step":
        head = (2 if case["audio2"] else case["vocab"]) + (N_VQ * AUDIO_VOCAB if moss else 0)
        total["bytes"] += 2 * head * (HIDDEN + 1)
        total["flops"] += 2.0 * head * HIDDEN
    return total


def tolerance(case: dict) -> dict:
    if case["kind"] in ("op", "gptq"):
        return {"rel": 7e-3}
    if case["kind"] == "prompt":
        return {"rel": 2e-2}
    return {"rel": 0.1 if case["layers"] > 4 else 3e-2}
