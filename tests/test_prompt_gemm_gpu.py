"""GPU parity of the GEMM with dequantised operands on the reference's records
(``mtl_w4_gemm_prompt_qsz``) against float64, and the routes that take it.

fp32 output: the products are exact and the sums run in float32 over K, so the relative error
is a few times 2^-24 sqrt(K / 32) at most, with a margin 2e-6 at K <= 4608; bf16 output adds
its rounding, 2^-9 / sqrt(3) of each value (relative 2-norm 1.7e-3, bar 2.5e-3).
"""
import ctypes

import pytest
import torch

from moss_tts_lite_amd import _native as N
from moss_tts_lite_amd import ops

pytestmark = pytest.mark.gpu


def record(dev, n, k, g, seed, s_exp=0):
    gen = torch.Generator(device=dev).manual_seed(seed)
    q = torch.randint(0, 16, (n, k), device=dev, generator=gen)
    pre = (q[:, 1::2] | (q[:, 0::2] << 4)).to(torch.uint8)
    s = torch.rand(k // g, n, device=dev, generator=gen) * 0.004 + 0.002
    z = torch.randn(k // g, n, device=dev, generator=gen) * 0.002
    qsz = (torch.stack([s, z], -1) * 2.0 ** s_exp).bfloat16()
    sc, zr = (qsz[..., i].t().double().repeat_interleave(g, 1) for i in (0, 1))
    return ops.convert_weight_to_int4pack(pre.contiguous(), 8), qsz, (q.double() - 8) * sc + zr


def workspace(m, k, n, g, dev):
    t, c = (m + 15) // 16, -(-(k // g) // 32)
    return torch.empty(t * (k // 32 + 3 * c) * 1024 + n // 16 * c * 1024 + k // g * n * 2 + 16
                       + 64 * t + 4 * n, dtype=torch.uint8, device=dev)


def run(x, packed, qsz, g, epilogue, y, ldx=None):
    m, k = x.shape
    n = qsz.shape[1]
    ws = workspace(m, k, n, g, x.device)
    N.check(N.load().mtl_w4_gemm_prompt_qsz(
        x.data_ptr(), m, x.stride(0), k, packed.data_ptr(), qsz.data_ptr(), n, g, epilogue,
        N.OUT_F32 if y.dtype == torch.float32 else N.OUT_BF16, y.data_ptr(), y.stride(0),
        ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream), "prompt gemm")
    torch.cuda.synchronize()
    return y


def rel(a, b):
    return float((a.double() - b).norm() / b.norm())


# every count of row tiles per workgroup (1 .. 6), a ragged last tile, ragged column tiles, one
# and several turns (K = 256: one block per wave group; 1792: 7 blocks), every group size
@pytest.mark.parametrize("m,k,n,g", [
    (1, 256, 16, 32), (16, 512, 256, 256), (17, 768, 272, 128), (33, 1792, 336, 64),
    (65, 1024, 1040, 32), (97, 4608, 256, 256), (389, 1024, 4096, 32), (600, 512, 5120, 128),
    (1100, 768, 4096, 64), (1536, 512, 4096, 128), (21, 16640, 64, 128),
    # grids of workgroups that take all of K (1.5 workgroups per CU and more): 2 and 6 blocks,
    # a ragged last column tile, 4, 5 and 6 row tiles
    (420, 256, 24592, 128), (200, 768, 24576, 64), (389, 512, 24576, 32), (576, 256, 18432, 256),
])
def test_prompt_gemm_matches_float64(dev, m, k, n, g):
    packed, qsz, w = record(dev, n, k, g, m + k + n)
    gen = torch.Generator(device=dev).manual_seed(7)
    xb = torch.randn(m, k + 8, device=dev, generator=gen)
    xb[:, ::37] *= 50.0
    x = xb.bfloat16()[:, :k]                     # a row pitch of its own
    ref = x.double() @ w.t()
    y = run(x, packed, qsz, g, N.EPI_NONE, torch.empty(m, n, device=dev))
    assert rel(y, ref) < 2e-6
    # rows 4 bytes off a 16-byte pitch: the unpacked stores
    wide = torch.zeros(m, n + 1, device=dev)
    assert torch.equal(run(x, packed, qsz, g, N.EPI_NONE, wide[:, :n]), y) and not wide[:, n:].any()
    yb = run(x, packed, qsz, g, N.EPI_NONE, torch.empty(m, n, device=dev, dtype=torch.bfloat16))
    assert torch.equal(yb, y.bfloat16())
    h = torch.randn(m, n, device=dev, generator=gen).bfloat16()
    hr = (y.bfloat16().float() + h.float()).bfloat16()
    assert torch.equal(run(x, packed, qsz, g, N.EPI_RESIDUAL, h), hr)
    if n % 64 == 0:
        act = run(x, packed, qsz, g, N.EPI_SILU_MUL,
                  torch.empty(m, n // 2, device=dev, dtype=torch.bfloat16))
        gu = y.bfloat16().float().reshape(m, n // 64, 2, 32)
        want = torch.nn.functional.silu(gu[:, :, 0]).bfloat16().float() * gu[:, :, 1]
        # the hardware exp and reciprocal: one bf16 ulp where the quotient is near a boundary
        assert rel(act, want.reshape(m, -1).double()) < 2.5e-3


def test_prompt_gemm_ranges(dev):
    # scales and activations far from 1, an all-zero row and an all-zero column: the powers of
    # two found per row and column keep the operands in f16's range; a row with an infinity is
    # not finite and leaves the others alone
    m, k, n, g = 70, 1024, 512, 64
    gen = torch.Generator(device=dev).manual_seed(3)
    base = torch.randn(m, k, device=dev, generator=gen)
    for x_exp, s_exp in ((0, 0), (60, -60), (-70, 40), (30, 10), (-40, -40)):
        packed, qsz, w = record(dev, n, k, g, 5, s_exp)
        qsz[:, 3] = 0
        w[3] = 0
        x = (base * 2.0 ** x_exp).bfloat16()
        x[11] = 0
        y = run(x, packed, qsz, g, N.EPI_NONE, torch.empty(m, n, device=dev))
        ref = x.double() @ w.t()
        assert rel(y, ref) < 2e-6 and not y[11].any() and not y[:, 3].any()
        xi = x.clone()
        xi[5, 100] = float("inf")
        yi = run(xi, packed, qsz, g, N.EPI_NONE, torch.empty(m, n, device=dev))
        keep = torch.arange(m, device=dev) != 5
        assert torch.equal(yi[keep], y[keep]) and not torch.isfinite(yi[5, :3]).any()


def test_prompt_gemm_checks(dev):
    packed, qsz, _ = record(dev, 256, 512, 32, 1)
    x = torch.zeros(20, 512, device=dev, dtype=torch.bfloat16)
    y = torch.empty(20, 256, device=dev, dtype=torch.bfloat16)
    ws = workspace(20, 512, 256, 32, dev)

    def call(m=20, k=512, n=256, g=32, epi=0, wsn=ws.numel(), ldy=256):
        return N.load().mtl_w4_gemm_prompt_qsz(
            x.data_ptr(), m, 512, k, packed.data_ptr(), qsz.data_ptr(), n, g, epi, N.OUT_BF16,
            y.data_ptr(), ldy, ws.data_ptr(), wsn, torch.cuda.current_stream().cuda_stream)

    assert call() == 0
    torch.cuda.synchronize()
    for bad in (dict(m=0), dict(k=384), dict(n=248), dict(g=48), dict(epi=9), dict(ldy=128),
                dict(wsn=ws.numel() - 64)):
        assert call(**bad) < 0, bad


@pytest.mark.parametrize("m,k,n,g", [(300, 1024, 2000, 32), (389, 4096, 24576, 32), (700, 4096, 6144, 64)])
def test_int4pack_mm_route(dev, m, k, n, g):
    # the drop-in takes this GEMM for many rows: the same bits, also replayed from a graph
    assert N.load().mtl_w4_gemm_prompt_qsz_workspace_bytes(m, k, n, g) > 0
    packed, qsz, w = record(dev, n, k, g, 9)
    x = torch.randn(m, k, device=dev).bfloat16()
    y = ops.weight_int4pack_mm(x, packed, g, qsz)
    want = run(x, packed, qsz, g, N.EPI_NONE, torch.empty_like(y))
    assert torch.equal(y, want) and rel(y, x.double() @ w.t()) < 2.5e-3
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.weight_int4pack_mm(x, packed, g, qsz)
    for i in range(3):
        x.copy_(torch.randn(m, k, device=dev).bfloat16())
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ops.weight_int4pack_mm(x, packed, g, qsz)), i


def test_embed_rows_unaligned_table(dev):
    # 11 tables (more than one set of 8), one of them 2 bytes off a 16-byte boundary
    hidden, rows = 72, 5
    gen = torch.Generator(device=dev).manual_seed(2)
    store = [torch.randn(30 * hidden + 1, device=dev, generator=gen).bfloat16() for _ in range(11)]
    tabs = [t[(1 if i == 4 else 0):][:30 * hidden].reshape(30, hidden) for i, t in enumerate(store)]
    ids = torch.randint(-1, 31, (rows, 11), device=dev, generator=gen)
    ptrs = torch.tensor([t.data_ptr() for t in tabs], dtype=torch.int64, device=dev)
    vocabs = torch.full((11,), 30, dtype=torch.int64, device=dev)
    out = torch.empty(rows, hidden, dtype=torch.bfloat16, device=dev)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    N.check(N.load().mtl_embed_rows(ids.data_ptr(), rows, 11, ptrs.data_ptr(), vocabs.data_ptr(),
                                    hidden, out.data_ptr(), st), "embed rows")
    torch.cuda.synchronize()
    for r in range(rows):
        h = None
        for t, i in zip(tabs, ids[r].tolist()):
            v = t[i] if 0 <= i < 30 else torch.zeros_like(t[0])
            h = v if h is None else h + v
        assert torch.equal(out[r], h)


@pytest.mark.parametrize("m,k,n,g,act", [
    (17, 512, 128, 32, True), (40, 768, 256, 256, True), (65, 4096, 384, 64, True),
    (200, 1024, 1024, 128, True), (33, 12288, 128, 128, True), (100, 1024, 256, 128, False),
])
def test_gptq_module_prompt_rows(dev, m, k, n, g, act):
    # more than 16 rows run on the prompt-length GEMM: against float64, equal to the C entry on
    # the gathered x, for a strided batch, and inside a graph captured before the first call
    from moss_tts_lite_amd.gptq import GPTQLinear
    from oracle import synth
    from tests.test_gemm_gpu import TOL_F32, rel_l2, t_bf16, t_f16, t_i32

    case = synth.gptq_case(k=k, n=n, m=m, group=g, act_order=act, seed=m + k + n)

    def linear():
        return GPTQLinear.from_buffers(t_i32(case["qweight"], dev), t_i32(case["qzeros"], dev),
                                       t_f16(case["scales"], dev),
                                       t_i32(case["g_idx"], dev) if act else None, g).post_init()

    lin, x = linear(), t_bf16(case["x_bits"], dev)
    y = lin(x, out_dtype=torch.float32)
    assert rel_l2(y.cpu().numpy(), case["y_ref"]) < TOL_F32
    xg = x if lin.perm is None else x.index_select(1, lin.perm.long())
    sc, qz = lin.strip_meta()
    assert torch.equal(y, ops.prefill_gemm(xg, lin._strip, sc, qz, n, g, out_dtype=torch.float32))
    wide = torch.zeros(m, k + 3, dtype=torch.bfloat16, device=dev)
    wide[:, 1:k + 1] = x
    assert torch.equal(lin(wide[:, 1:k + 1], out_dtype=torch.float32), y)
    assert lin(x.reshape(1, m, k)).shape == (1, m, n)
    fresh = linear()                              # captured before any eager call
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fresh(x, out_dtype=torch.float32)
    assert fresh._strip is None
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        assert rel_l2(out.cpu().numpy(), case["y_ref"]) < TOL_F32
        assert torch.equal(fresh(x, out_dtype=torch.float32), y)


def row_blocks(m, n, cus=256):
    """(row tiles per workgroup, workgroups) as the launch chooses them: the rounds over the CUs
    times the time of a turn at that many row tiles."""
    tiles, ctiles, best, cost = -(-m // 16), -(-n // 256), 0, 0.0
    for nb in range(-(-tiles // 6), tiles + 1):
        rt = -(-tiles // nb)
        c = -(-nb * ctiles // cus) * (2.3 if rt <= 4 else 2.7 if rt == 5 else 3.1)
        if not best or c < cost:
            best, cost = nb, c
        if rt <= 4:
            break
    return -(-tiles // best), best * ctiles


# every kernel instance: 4, 5 and 6 row tiles (at 3 and 4 also fewer than the instance holds), one
# metadata record per block or two or four (g 128 / 256, 64, 32), K in halves or whole; K = 256
# and 768 are one and three blocks of a half, two and six whole
_INSTANCES = [(m, n, two, rt) for two, shapes in ((True, ((49, 256, 4), (80, 33024, 5), (89, 33040, 6))),
                                                  (False, ((40, 98304, 4), (208, 33024, 5),
                                                           (251, 33040, 6))))
              for m, n, rt in shapes]


@pytest.mark.parametrize("g", [32, 64, 128, 256])
@pytest.mark.parametrize("m,n,two,rt", _INSTANCES)
def test_prompt_gemm_every_instance(dev, m, n, two, rt, g):
    tiles, groups = row_blocks(m, n)
    assert max(tiles, 4) == rt and (2 * groups < 3 * 256) == two
    for k in (256, 768) if n < 1000 else (256,):
        packed, qsz, w = record(dev, n, k, g, m + g)
        x = torch.randn(m, k, device=dev, generator=torch.Generator(device=dev).manual_seed(n)).bfloat16()
        y = run(x, packed, qsz, g, N.EPI_NONE, torch.empty(m, n, device=dev))
        ref = x.double() @ w.t()
        assert rel(y, ref) < 2e-6
        # each row tile and the last, ragged column tile by themselves
        err = [float((a - b).norm() / b.norm()) for a, b in zip(y.double().split(16), ref.split(16))]
        assert max(err) < 4e-6 and rel(y[:, n // 256 * 256 - 256:], ref[:, n // 256 * 256 - 256:]) < 4e-6
        if n % 64 == 0:
            act = run(x, packed, qsz, g, N.EPI_SILU_MUL,
                      torch.empty(m, n // 2, device=dev, dtype=torch.bfloat16))
            gu = y.bfloat16().float().reshape(m, n // 64, 2, 32)
            want = torch.nn.functional.silu(gu[:, :, 0]).bfloat16().float() * gu[:, :, 1]
            assert rel(act, want.reshape(m, -1).double()) < 2.5e-3
        h = torch.randn(m, n, device=dev).bfloat16()
        hr = (y.bfloat16().float() + h.float()).bfloat16()
        assert torch.equal(run(x, packed, qsz, g, N.EPI_RESIDUAL, h), hr)


def moss_backbone(dev, hidden, inter, g, max_seq, keep_up):
    """Two layers of the reference's records with v_proj in bf16 and, with ``keep_up``, up_proj
    of the first."""
    from moss_tts_lite_amd import model
    from moss_tts_lite_amd.gptq import QszLinear, interleave_qsz_gate_up
    gen = torch.Generator(device=dev).manual_seed(hidden + inter)
    heads, kv = hidden // 128, max(hidden // 512, 1)
    randn = lambda *s, std=1.0: (torch.randn(*s, device=dev, generator=gen) * std).bfloat16()  # noqa: E731
    norm = lambda n: (1 + 0.05 * torch.randn(n, device=dev, generator=gen)).bfloat16()  # noqa: E731

    def lin(n, k, seed):
        packed, qsz, _ = record(dev, n, k, g, seed)
        return QszLinear(packed, qsz, g)

    layers = []
    for i in range(2):
        lw = {"input_layernorm": norm(hidden), "post_attention_layernorm": norm(hidden),
              "q_norm": norm(128), "k_norm": norm(128), "qkv": lin((heads + kv) * 128, hidden, 10 * i),
              "v": randn(kv * 128, hidden, std=0.02), "o": lin(hidden, hidden, 10 * i + 1),
              "down": lin(hidden, inter, 10 * i + 2)}
        gate, up = lin(inter, hidden, 10 * i + 3), lin(inter, hidden, 10 * i + 4)
        if keep_up and i == 0:
            lw.update(gate=gate, up=randn(inter, hidden, std=0.02))
        else:
            lw["gate_up"] = interleave_qsz_gate_up(gate, up)
        layers.append(lw)
    cfg = model.BackboneConfig(hidden=hidden, n_heads=heads, n_kv_heads=kv, head_dim=128,
                               intermediate=inter, n_layers=2, vocab=64, group_size=g,
                               act_order=False, max_seq=max_seq, n_vq=2, audio_vocab=33,
                               audio_pad_code=32, two_way_ids=(0, 1))
    return model.Int4Backbone(cfg, {
        "layers": layers, "embed_tokens": randn(64, hidden), "final_norm": norm(hidden),
        "head": randn(64, hidden, std=0.02), "emb_ext": list(randn(2, 33, hidden, std=0.2)),
        "head_audio": randn(2, 33, hidden, std=0.02)})


# the full width at a length where every linear takes this GEMM by itself, and small layers where
# it is made to: all of them, and each alone (plain x into one GEMM, staged x into the next)
@pytest.mark.parametrize("hidden,inter,rows,only", [
    (4096, 12288, 1100, "rule"), (512, 1024, 70, "all"), (512, 1024, 70, "qkv"),
    (512, 1024, 70, "o"), (512, 1024, 70, "gate_up"), (512, 1024, 70, "down")])
@pytest.mark.parametrize("keep_up", [False, True])
def test_prompt_layers_on_this_gemm(dev, monkeypatch, hidden, inter, rows, only, keep_up):
    # kept v_proj on plain x, the residual into h before the next norm, SiLU*up, the last layer's
    # down, kept up_proj: against the same layers on the prompt-length GEMM
    from moss_tts_lite_amd.fast import FastMossDecoder
    model = moss_backbone(dev, hidden, inter, 32, rows + 8, keep_up)
    dec = FastMossDecoder(model)
    gen = torch.Generator(device=dev).manual_seed(rows)
    ids = torch.stack([torch.randint(0, n, (rows,), device=dev, generator=gen)
                       for n in (64, 33, 33)], 1)
    names = {id(lyr[k]): k for lyr in model.layers for k in ("qkv", "o", "gate_up", "down")}
    asked = set()

    def wide_bytes(self, m, lin):
        if only not in ("all", names[id(lin)]):
            return 0
        asked.add(names[id(lin)])
        return workspace(m, lin.in_features, lin.out_features, lin.group_size, "meta").numel()

    def prompt():
        model.reset_cache()
        h = dec.prefill_rows(ids).clone()
        return h, model.k_cache[:, :, :rows].clone(), model.v_cache[:, :, :rows].clone()

    if only == "rule":
        dec._prefill_io(rows)
        assert all(dec._wide_bytes(rows, lyr[k]) for lyr in model.layers
                   for k in ("qkv", "o", "gate_up", "down") if not (keep_up and k == "gate_up"))
    else:
        monkeypatch.setattr(FastMossDecoder, "_wide_bytes", wide_bytes)
    got = prompt()
    assert only == "rule" or asked == ({only} if only != "all" else {"qkv", "o", "gate_up", "down"})
    monkeypatch.setattr(FastMossDecoder, "_wide_bytes", lambda self, m, lin: 0)
    want = prompt()
    # the two differ by fp32 rounding before each of about seven bf16 roundings a layer (2^-9 /
    # sqrt(3) where one flips): below sqrt(2 * 7 * 2) * 1.1e-3 = 6e-3 over two layers
    for a, b in zip(got, want):
        assert torch.isfinite(a).all() and rel(a.float(), b.double()) < 6e-3
    # layer 0's value rows come from the bf16 v_proj on the same normed rows
    assert torch.equal(got[2][0], want[2][0])


@pytest.mark.parametrize("zero_offset", [0, 1])
@pytest.mark.parametrize("act", [True, False])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_gptq_module_route_against_split_k(dev, zero_offset, act, dt):
    # the new route of many rows against the split-K GEMM over what a module takes: both zero
    # conventions and output types, x 2 bytes off a 16-byte boundary, transposed, expanded, with
    # leading dimensions, the row counts around 16, a tile and two of them
    from moss_tts_lite_amd.gptq import GPTQLinear
    from oracle import synth
    from tests.test_gemm_gpu import t_bf16, t_f16, t_i32

    k, n, g = 768, 256, 64
    case = synth.gptq_case(k=k, n=n, m=130, group=g, act_order=act, seed=31 + zero_offset)
    lin = GPTQLinear.from_buffers(t_i32(case["qweight"], dev), t_i32(case["qzeros"], dev),
                                  t_f16(case["scales"], dev),
                                  t_i32(case["g_idx"], dev) if act else None, g,
                                  zero_offset=zero_offset).post_init()
    x = t_bf16(case["x_bits"], dev)
    w = lin.dequantize().double()
    off = torch.cat([x.new_zeros(1), x.reshape(-1)])[1:].reshape(130, k)
    forms = [x[:m] for m in (15, 16, 17, 63, 64, 65, 130)]
    forms += [off, x[:64].t().contiguous().t(), x[:1].expand(40, k), x[:120].reshape(2, 3, 20, k)]
    qw, qz, sc, perm = lin.kernel_args()
    for xf in forms:
        y = lin(xf, out_dtype=dt)
        old = ops.gptq_gemm(xf.clone(memory_format=torch.contiguous_format), qw, qz, sc, g,
                            perm=perm, zero_offset=zero_offset, out_dtype=dt)
        ref = xf.double() @ w
        assert y.shape == old.shape == ref.shape and y.dtype == dt
        # 32-bit sums in another order, or those rounded to bf16 (2^-9 / sqrt(3) of each value)
        bar = 4e-6 if dt == torch.float32 else 2.5e-3
        assert rel(y, ref) < bar and rel(y, ref) < 2 * rel(old, ref) + 1e-7
