"""Decode attention over caches of more than 4096 positions (chunks of several blocks): against
float64, the fused form against the two-kernel form bit for bit, both hand-offs."""
import ctypes

import pytest
import torch

from moss_tts_lite_amd import _native as N

pytestmark = pytest.mark.gpu


# the edges of a block and of the first 64 blocks, a chunk's third block, a ragged cache end
@pytest.mark.parametrize("H,Hkv,max_seq,positions", [
    (32, 8, 8192, (0, 63, 64, 4095, 4096, 4097, 4159, 4160, 6000, 8191)),
    (32, 8, 9000, (4100, 8191, 8192, 8255, 8999)),
    (8, 2, 4200, (4000, 4095, 4096, 4199)),      # agent-scope hand-off
])
@pytest.mark.parametrize("local", [1, 0])
def test_long_cache_attention(dev, H, Hkv, max_seq, positions, local):
    lib = N.load()
    gen = torch.Generator(device=dev).manual_seed(max_seq)
    ncols, splits = (H + 2 * Hkv) * 128, 2
    cache = torch.randn(2, Hkv, max_seq, 128, device=dev, generator=gen).bfloat16()
    qn, kn = (1 + 0.1 * torch.randn(128, device=dev, generator=gen).bfloat16() for _ in range(2))
    ang = torch.rand(max_seq, 64, device=dev, generator=gen) * 6.28
    cos, sin = (torch.cat([f(ang)] * 2, -1).bfloat16() for f in (torch.cos, torch.sin))
    ws = torch.zeros(int(lib.mtl_decode_attention_workspace_bytes(H, 128)), dtype=torch.uint8,
                     device=dev)
    idx = torch.randperm(H * 128, device=dev, generator=gen).int()
    scale, eps = ctypes.c_float(128 ** -0.5), ctypes.c_float(1e-6)
    st = torch.cuda.current_stream().cuda_stream
    try:
        assert lib.mtl_decode_attention_set_handoff(local) == 0
        for pos in positions:
            parts = torch.randn(splits, ncols, device=dev, generator=gen)
            tpos = torch.tensor([pos], dtype=torch.int64, device=dev)
            res = []
            for fused in (False, True):
                kc, vc = cache[0].clone(), cache[1].clone()
                out = torch.zeros(H * 128, dtype=torch.bfloat16, device=dev)
                if fused:
                    N.check(lib.mtl_decode_attention_fused(
                        parts.data_ptr(), splits, qn.data_ptr(), kn.data_ptr(), cos.data_ptr(),
                        sin.data_ptr(), kc.data_ptr(), vc.data_ptr(), tpos.data_ptr(),
                        out.data_ptr(), idx.data_ptr(), H, Hkv, 128, max_seq, scale, eps,
                        ws.data_ptr(), ws.numel(), st), "attention fused")
                else:
                    q = torch.zeros(H * 128, dtype=torch.bfloat16, device=dev)
                    N.check(lib.mtl_qk_norm_rope_kv_partials(
                        parts.data_ptr(), splits, qn.data_ptr(), kn.data_ptr(), cos.data_ptr(),
                        sin.data_ptr(), tpos.data_ptr(), q.data_ptr(), kc.data_ptr(),
                        vc.data_ptr(), H, Hkv, 128, max_seq, eps, st), "qk rope")
                    N.check(lib.mtl_decode_attention(
                        q.data_ptr(), kc.data_ptr(), vc.data_ptr(), tpos.data_ptr(),
                        out.data_ptr(), idx.data_ptr(), H, Hkv, 128, max_seq, scale,
                        ws.data_ptr(), ws.numel(), st), "attention")
                res.append((out, kc, vc))
            assert all(torch.equal(a, b) for a, b in zip(*res)), pos
            k, v = (c[:, :pos + 1].double().repeat_interleave(H // Hkv, 0) for c in res[0][1:])
            s = torch.einsum("hd,hpd->hp", q.double().reshape(H, 128), k) * 128 ** -0.5
            ref = torch.einsum("hp,hpd->hd", torch.softmax(s, -1), v).reshape(-1)
            got = res[0][0].double()[idx.long()]
            # bf16 probabilities and output: 2^-9 each, relative to values that average out
            assert float((got - ref).norm() / ref.norm()) < 1e-2, pos
            assert not ws[:1024].any()           # counters back at zero, placement held
    finally:
        lib.mtl_decode_attention_set_handoff(1)


# row blocks past one and two turns of the deal (32 blocks of 16 rows), a ragged last block, both
# group counts (4 and 8 q heads per kv head), fewer tiles than wave groups
@pytest.mark.parametrize("H,Hkv,L,pos0", [(8, 2, 530, 0), (4, 1, 1100, 3), (16, 2, 545, 0),
                                          (8, 2, 19, 61), (4, 4, 65, 0)])
def test_prefill_attention_rows(dev, H, Hkv, L, pos0):
    gen = torch.Generator(device=dev).manual_seed(L)
    S = pos0 + L + 5
    kc, vc = (torch.randn(Hkv, S, 128, device=dev, generator=gen).bfloat16() for _ in range(2))
    kc[:, S - 5:] = float("nan")                 # rows past the prompt are not read into a result
    vc[:, S - 5:] = float("nan")
    q = torch.randn(L, H * 128, device=dev, generator=gen).bfloat16()
    out = torch.zeros(L, H * 128, dtype=torch.bfloat16, device=dev)
    N.check(N.load().mtl_prefill_attention(
        q.data_ptr(), kc.data_ptr(), vc.data_ptr(), L, pos0, out.data_ptr(), H * 128, None, H, Hkv,
        128, S, ctypes.c_float(128 ** -0.5), torch.cuda.current_stream().cuda_stream), "attention")
    torch.cuda.synchronize()
    n = pos0 + L
    k, v = (c[:, :n].double().repeat_interleave(H // Hkv, 0) for c in (kc, vc))
    s = q.double().reshape(L, H, 128).transpose(0, 1) @ k.transpose(1, 2) * 128 ** -0.5
    keep = torch.arange(n, device=dev)[None] <= pos0 + torch.arange(L, device=dev)[:, None]
    ref = (torch.softmax(s.masked_fill(~keep, float("-inf")), -1) @ v).transpose(0, 1).reshape(L, -1)
    err = (out.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) < 1e-2               # bf16 probabilities and output
    # through an output index, 16-byte aligned and not, and with rows 2 bytes off: the same values
    perm = torch.randperm(H * 128, device=dev, generator=gen).int()
    for ix, ld, off in ((perm, None, 0), (None, H * 128 + 1, 1),
                        (torch.cat([perm[:1], perm])[1:], None, 0)):
        ld = ld or H * 128
        buf = torch.zeros(L * ld + off, dtype=torch.bfloat16, device=dev)
        N.check(N.load().mtl_prefill_attention(
            q.data_ptr(), kc.data_ptr(), vc.data_ptr(), L, pos0, buf[off:].data_ptr(), ld,
            None if ix is None else ix.data_ptr(), H, Hkv, 128, S, ctypes.c_float(128 ** -0.5),
            torch.cuda.current_stream().cuda_stream), "attention")
        torch.cuda.synchronize()
        got = buf[off:].reshape(L, ld)[:, :H * 128]
        assert torch.equal(got if ix is None else got[:, ix.long()], out)
