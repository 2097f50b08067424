"""When a GPTQ linear's kernel copies are made, kept and made again: the module's own code on the
CPU, its kernels replaced by plain stand-ins that fill their outputs outside torch's sight, as
the library does through raw pointers."""
import ctypes
import io
import types

import pytest
import torch

from moss_tts_lite_amd import gptq, ops

K, N, G = 256, 128, 64


def _filled(src):
    """A copy that only memory knows of: torch sees an empty tensor."""
    src = src.contiguous()
    out = torch.empty_like(src)
    ctypes.memmove(out.data_ptr(), src.data_ptr(), src.numel() * src.element_size())
    return out


def _product(x, qw, qz, sc, g, perm, zo, dt):
    """x @ dequant(W) of AutoGPTQ-layout tensors, the weight's rows sorted by group."""
    j = torch.arange(8, dtype=torch.int32) * 4
    q = ((qw.unsqueeze(1) >> j.view(1, 8, 1)) & 15).reshape(-1, qw.shape[1]).float()
    z = ((qz.unsqueeze(2) >> j) & 15).reshape(qz.shape[0], -1).float() + zo
    w = (q - z.repeat_interleave(g, 0)) * sc.float().repeat_interleave(g, 0)
    xg = x if perm is None else x.index_select(-1, perm.long())
    return (xg.float() @ w).to(dt)


@pytest.fixture
def kernels(monkeypatch):
    """The stand-ins and the list of products that ran."""
    ran = []

    def strip(name):
        def run(x, w, sc, qz, n, g, zo=0, perm=None, dt=torch.bfloat16):
            ran.append(name)
            if name == "rows":
                sc, qz = qz, sc
            return _product(x, w, qz, sc, g, perm, zo, dt)
        return run

    def plain(x, qw, qz, sc, g, perm=None, zo=0, dt=torch.bfloat16):
        ran.append("gptq")
        return _product(x, qw, qz, sc, g, perm, zo, dt)

    def actorder(qw, g_idx, g):
        if g_idx.numel() != qw.shape[0] * 8:
            raise RuntimeError("g_idx must have K entries")
        perm = torch.argsort(g_idx, stable=True).int()
        j = torch.arange(8, dtype=torch.int32) * 4
        q = ((qw.unsqueeze(1) >> j.view(1, 8, 1)) & 15).reshape(-1, qw.shape[1])[perm.long()]
        return _filled((q.view(-1, 8, qw.shape[1]) << j.view(1, 8, 1)).sum(1).int()), _filled(perm)

    lib = types.SimpleNamespace(gptq_gemm=plain, strip_gemv=strip("gemv"),
                                strip_rows_gemm=strip("rows"), prompt_gemm=strip("prompt"))
    stream = types.SimpleNamespace(synchronize=lambda: None)
    monkeypatch.setattr(ops, "torch_ops", lambda: lib)
    monkeypatch.setattr(ops, "overload", lambda name: getattr(lib, name))
    monkeypatch.setattr(ops, "strip_weights", _filled)
    monkeypatch.setattr(ops, "strip_meta", lambda sc, qz, g: (_filled(sc), _filled(qz)))
    monkeypatch.setattr(ops, "actorder_prepare", actorder)
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda t: True), raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: stream)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    return ran


def _buffers(seed, act):
    gen = torch.Generator().manual_seed(seed)
    g_idx = torch.arange(K, dtype=torch.int32) // G
    return (torch.randint(-2**31, 2**31 - 1, (K // 8, N), dtype=torch.int32, generator=gen),
            torch.randint(-2**31, 2**31 - 1, (K // G, N // 8), dtype=torch.int32, generator=gen),
            (torch.rand(K // G, N, generator=gen) * 0.01 + 0.01).half(),
            g_idx[torch.randperm(K, generator=gen)] if act else None)


def _linear(seed, act):
    return gptq.GPTQLinear.from_buffers(*_buffers(seed, act), G).post_init()


def _x(m):
    return torch.randn(m, K, generator=torch.Generator().manual_seed(m)).bfloat16()


ROWS = (1, 4, 40)            # the strip GEMV, the skinny GEMM, the prompt-length GEMM


@pytest.mark.parametrize("act", [False, True])
def test_buffers_changed_after_use(kernels, act):
    # a linear that has run follows its buffers as a new one does: load_state_dict, an in-place
    # change of the metadata, replaced tensors
    for m in ROWS:
        x = _x(m)
        lin = _linear(1, act)
        first = lin(x)
        lin.load_state_dict(_linear(2, act).state_dict())
        assert torch.equal(lin(x), _linear(2, act)(x)) and not torch.equal(lin(x), first)
        lin.scales.mul_(2)
        assert torch.allclose(lin(x).float(), 2 * _linear(2, act)(x).float(), rtol=1e-2)
        third = _linear(3, act)
        lin.qweight, lin.qzeros, lin.scales, lin.g_idx = (t.clone() for t in (
            third.qweight, third.qzeros, third.scales, third.g_idx))
        assert torch.equal(lin(x), third(x)), m
    assert set(kernels) == {"gemv", "rows", "prompt"}


def test_post_init_makes_every_copy_again(kernels):
    # after a write that torch does not count, here through .data
    for act in (False, True):
        lin, other = _linear(1, act), _linear(2, act)
        for m in ROWS:
            lin(_x(m))
        for a, b in zip(lin.buffers(), other.buffers()):
            a.data.copy_(b)
        lin.post_init()
        assert all(torch.equal(lin(_x(m)), other(_x(m))) for m in ROWS)


def test_copies_are_made_again_in_place(kernels):
    # a captured graph or a decoder that holds a copy's address reads the new weight through it
    lin = _linear(1, True)
    for m in ROWS:
        lin(_x(m))
    at = [t.data_ptr() for t in (lin._kernel_qweight, lin._perm, lin._strip, *lin._strip_meta)]
    lin.load_state_dict(_linear(2, True).state_dict())
    y = [lin(_x(m)) for m in ROWS]
    new = [t.data_ptr() for t in (lin._kernel_qweight, lin._perm, lin._strip, *lin._strip_meta)]
    assert at == new and all(torch.equal(a, _linear(2, True)(_x(m))) for a, m in zip(y, ROWS))
    made = lin._strip
    lin(_x(40))
    assert lin._strip is made


def test_a_decoder_reads_the_copies_as_they_are(kernels):
    # made at the first request, at the same addresses after a change that a call has followed
    lin = _linear(1, True)
    args = lin.strip_args()
    assert args == lin.stream_weight(True) + lin.strip_meta()
    lin.load_state_dict(_linear(2, True).state_dict())
    assert lin.strip_args()[0] is args[0] and torch.equal(args[0], _linear(1, True).strip_args()[0])
    lin(_x(40))
    new = _linear(2, True).strip_args()
    assert all(torch.equal(args[i], new[i]) for i in (0, 2, 3)) and lin.strip_args()[0] is args[0]


def test_dropped_and_reordered_weights_keep_their_copies(kernels):
    # after drop_original or keep_strip_only the copies are all there is of the weight; the
    # metadata still follows its buffers
    x, ref = _x(40), _linear(5, True)(_x(40))
    lin = _linear(5, True)
    lin(x)
    lin.drop_original()
    assert not lin.qweight.numel() and torch.equal(lin(x), ref)
    with pytest.raises(RuntimeError):
        lin.post_init()                              # nothing left to sort, nothing lost
    assert torch.equal(lin(x), ref)
    lin.reorder_output_columns(torch.arange(N).flip(0))
    assert torch.equal(lin(x), ref.flip(-1))
    lin.keep_strip_only()
    assert torch.equal(lin(x), ref.flip(-1))
    lin.scales.mul_(2)
    assert torch.allclose(lin(x).float(), 2 * ref.flip(-1).float(), rtol=1e-2)


def test_a_linear_on_the_host_is_refused():
    # no stand-ins: the copies' kernels take raw pointers and must not see host memory
    for act in (False, True):
        lin = gptq.GPTQLinear.from_buffers(*_buffers(1, act), G)
        for m in ROWS:
            with pytest.raises(RuntimeError, match="HIP device|'CPU' backend"):
                lin(_x(m))


def test_changed_inside_a_capture(kernels, monkeypatch):
    # nothing is kept that only a replay would fill: without act-order the call reads the buffers
    # or a copy of its own, with it the prepared weight is missing and the call is refused; a
    # change of the metadata alone needs no weight
    for act in (False, True):
        lin = _linear(1, act)
        for m in ROWS:
            lin(_x(m))
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
        strip, meta = lin._strip.clone(), lin._strip_meta[0].clone()
        lin.scales.mul_(2)
        ref = gptq.GPTQLinear.from_buffers(*_buffers(1, act), G)
        ref.scales.mul_(2)
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
        want = [ref(_x(m)) for m in ROWS]
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
        assert all(torch.equal(lin(_x(m)), w) for m, w in zip(ROWS, want))
        lin.load_state_dict(_linear(2, act).state_dict())
        for m in ROWS:
            if act:
                with pytest.raises(RuntimeError, match="before capturing"):
                    lin(_x(m))
            else:
                assert torch.equal(lin(_x(m)), _linear(2, act)(_x(m)))
        assert torch.equal(lin._strip, strip) and torch.equal(lin._strip_meta[0], meta)
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
        assert all(torch.equal(lin(_x(m)), _linear(2, act)(_x(m))) for m in ROWS)


@pytest.mark.parametrize("act", [False, True])
@pytest.mark.parametrize("m", ROWS)
def test_traced_before_any_call(kernels, act, m):
    # a trace records torch's operations only: a copy that a kernel fills would be recorded as an
    # uninitialised tensor, so none is made there and the buffers' own product is recorded
    from torch.fx.experimental.proxy_tensor import make_fx
    x, want = _x(m), _linear(1, act)(_x(m))
    lin = _linear(1, act)
    traced = torch.jit.trace(lin, x, check_trace=False)
    assert lin._strip is None and lin._strip_meta is None
    assert torch.equal(traced(x), want)
    for pre in (False, True):
        lin = _linear(1, act)
        fx = make_fx(lambda t: lin(t), pre_dispatch=pre)(x)
        assert lin._strip is None and torch.equal(fx(x), want)
    lin = _linear(1, act)
    rows = x.expand(2, m, K)
    assert torch.equal(torch.func.vmap(lin)(rows)[1], want)
    # the buffers of a linear that has run stay the traced graph's inputs for many rows
    if m > 16:
        lin(x)
        traced = torch.jit.trace(lin, x, check_trace=False)
        lin.scales.mul_(2)
        assert torch.allclose(traced(x).float(), 2 * want.float(), rtol=1e-2)


def test_traced_after_a_change(kernels):
    # without act-order the buffers are read; with it the sorted weight would have to be made
    # inside the trace (torch.jit.trace reads the module's properties first, which does it)
    from torch.fx.experimental.proxy_tensor import make_fx
    for act in (False, True):
        for m in ROWS:
            x, want = _x(m), _linear(2, act)(_x(m))
            lin = _linear(1, act)
            lin(x)
            lin.load_state_dict(_linear(2, act).state_dict())
            if act:
                with pytest.raises(RuntimeError, match="or tracing"):
                    make_fx(lambda t: lin(t))(x)
            else:
                assert torch.equal(make_fx(lambda t: lin(t))(x)(x), want)
            assert torch.equal(torch.jit.trace(lin, x, check_trace=False)(x), want)


@pytest.mark.parametrize("act", [False, True])
def test_first_call_inside_a_capture(kernels, monkeypatch, act):
    # what a capture makes is filled at replay and lives in the graph's memory: it is used there
    # and not kept, so an eager call before any replay reads copies of its own
    for m in (1, 4):
        lin, x = _linear(1, act), _x(m)
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
        lin(x)
        assert all(c is None for c in (lin._strip, lin._strip_meta, lin._perm16, lin._one_row))
        with pytest.raises(RuntimeError, match="capture"):
            lin.keep_strip_only()
        assert lin.qweight.numel()
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
        assert torch.equal(lin(_x(40)), _linear(1, act)(_x(40)))


def test_copies_are_waited_for(kernels, monkeypatch):
    # whichever call makes a copy, or makes it again, waits for it: the next may run on another
    # stream
    waits = []
    stream = types.SimpleNamespace(synchronize=lambda: waits.append(1))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: stream)
    for m in ROWS:
        lin = _linear(1, True)
        waits.clear()
        lin(_x(m))
        assert waits
        waits.clear()
        lin(_x(m))
        assert not waits
        lin.load_state_dict(_linear(2, True).state_dict())
        lin(_x(m))
        assert waits


def test_inference_tensors_are_read_at_every_call(kernels):
    # they keep no version, so a change in place leaves no mark: no copy of them is used for
    # the rows that were read from the buffers before there was one
    with torch.inference_mode():
        lin = _linear(1, False)
        x = _x(40)
        first = lin(x)
        lin.scales.mul_(2)
        assert torch.allclose(lin(x).float(), 2 * first.float(), rtol=1e-2)


def test_saved_modules(kernels):
    # with the copies and their marks, and as saved before there were marks
    lin = _linear(1, True)
    ref = [lin(_x(m)) for m in ROWS]
    for marked in (True, False):
        if not marked:
            del lin._src, lin._one_row
        buf = io.BytesIO()
        torch.save(lin, buf)
        buf.seek(0)
        back = torch.load(buf, weights_only=False)
        assert all(torch.equal(back(_x(m)), r) for m, r in zip(ROWS, ref))
        back.load_state_dict(_linear(2, True).state_dict())
        assert torch.equal(back(_x(40)), _linear(2, True)(_x(40)))


@pytest.mark.gpu
@pytest.mark.parametrize("act", [False, True])
def test_buffers_changed_after_use_on_the_device(dev, act):
    # the kernels themselves, eager and captured: a replay of many rows reads the buffers as
    # they are, of one row the copy that the eager call brought up to date
    def linear(seed):
        return gptq.GPTQLinear.from_buffers(*(None if b is None else b.to(dev)
                                              for b in _buffers(seed, act)), G).post_init()

    lin, other = linear(1), linear(2)
    want = {m: other(_x(m).to(dev)) for m in ROWS}
    graphs = {}
    for m in ROWS:
        x = _x(m).to(dev)
        lin(x)
        graphs[m] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graphs[m]):
            out = lin(x)
        graphs[m] = graphs[m], out, x
    lin.load_state_dict(other.state_dict())
    for m in ROWS:
        assert torch.equal(lin(_x(m).to(dev)), want[m]), m
    for _ in range(2):
        for m, (graph, out, x) in graphs.items():
            graph.replay()
            torch.cuda.synchronize()
            # the captured many-row call runs on the AutoGPTQ layout: other fp32 sums, bf16 out
            err = (out.float() - want[m].float()).norm() / want[m].float().norm()
            assert torch.equal(out, want[m]) if m <= 16 else float(err) < 4e-3, (m, float(err))


@pytest.mark.gpu
@pytest.mark.parametrize("act", [False, True])
@pytest.mark.parametrize("m", [1, 4])
def test_first_call_captured_on_the_device(dev, act, m):
    # a first call of one or few rows inside a capture, then an eager prompt before any replay,
    # on another stream: both right, and every replay
    def linear():
        return gptq.GPTQLinear.from_buffers(*(None if b is None else b.to(dev)
                                              for b in _buffers(1, act)), G).post_init()

    x, x40 = _x(m).to(dev), _x(40).to(dev)
    want, want40 = linear()(x), linear()(x40)
    lin = linear()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = lin(x)
    assert lin._strip is None
    other = torch.cuda.Stream()
    with torch.cuda.stream(other):
        assert torch.equal(lin(x40), want40)
    torch.cuda.synchronize()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(lin(x), want) and torch.equal(lin(x40), want40)
