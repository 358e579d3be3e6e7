"""The pipelined chunkwise kernel on q, k, v read in place from a projection's layout.

The strided call must be bit-equal to the call on contiguous copies (the same kernel, other addresses), over
head widths, ragged lengths, batches, the sequence split, f16, initial states, and views whose rows cannot be
read in place (odd row strides, an offset base), which take the copy; the C entry point itself against the contiguous
one, and the operator's memory, which shows whether it copied."""

import ctypes

import pytest
import torch

from helpers import dev

pytestmark = pytest.mark.gpu


def _views(B, NH, S, DQK, DV, dtype, layout, seed):
    g = torch.Generator().manual_seed(seed)
    out = []
    for D in (DQK, DQK, DV):
        t = torch.randn(B, S, NH, D, generator=g).to(dtype).to(dev())
        if layout == "odd_rows":      # rows NH * D + 4 apart: not 16-byte multiples
            big = torch.zeros(B, S, NH * D + 4, dtype=dtype, device=dev())
            big[..., :NH * D] = t.reshape(B, S, NH * D)
            t = big[..., :NH * D].unflatten(-1, (NH, D))
        elif layout == "offset":      # base 2 bytes past 16-byte alignment
            big = torch.zeros(t.numel() + 1, dtype=dtype, device=dev())
            big[1:] = t.reshape(-1)
            t = big[1:].view(B, S, NH, D)
        elif layout == "packed":      # slices of one fused projection
            big = torch.randn(B, S, 3, NH, D, generator=g).to(dtype).to(dev())
            t = big[:, :, 1]
        t = t.permute(0, 2, 1, 3)
        out.append(t[:, :1].expand(B, NH, S, D) if layout == "expanded" else t)
    q, k, v = out
    i = torch.randn(B, NH, S, generator=g).to(dtype).to(dev())
    f = (torch.randn(B, NH, S, generator=g) + 3).to(dtype).to(dev())
    return q, k, v, i, f


@pytest.mark.parametrize("B,NH,S,DQK,DV", [(1, 8, 100, 256, 512), (2, 4, 1000, 128, 256), (3, 2, 65, 96, 192), (1, 2, 1, 64, 64),
                                           (2, 1, 640, 192, 64), (1, 8, 2011, 256, 512)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["projection", "odd_rows", "offset", "packed", "expanded"])
def test_strided_equals_contiguous(gpu_case, B, NH, S, DQK, DV, dtype, layout):
    import xlstm_hip
    x = _views(B, NH, S, DQK, DV, dtype, layout, S)
    got = xlstm_hip.mlstm_chunkwise(*x, return_last_states=True, algo="pipelined")
    want = xlstm_hip.mlstm_chunkwise(*(t.contiguous() for t in x), return_last_states=True, algo="pipelined")
    for a, b in zip((got[0], *got[1]), (want[0], *want[1])):
        assert torch.equal(a, b)


def _strides(t):
    return [t.stride(0) if t.size(0) > 1 else 0, t.stride(1) if t.size(1) > 1 else 0, t.stride(2)]


@pytest.mark.parametrize("B,NH,S,DQK,DV", [(1, 8, 100, 256, 512), (2, 4, 1000, 128, 256), (3, 2, 65, 96, 192)])
@pytest.mark.parametrize("layout", ["projection", "packed", "expanded"])
def test_strided_entry_point(gpu_case, B, NH, S, DQK, DV, layout):
    from xlstm_hip import _lib
    lib = _lib.load()
    q, k, v, i, f = _views(B, NH, S, DQK, DV, torch.bfloat16, layout, S)
    ws_bytes = lib.xl_mlstm_chunkwise_workspace_size(B, NH, S, DQK, DV, 64, 1, 3)
    st = torch.cuda.current_stream().cuda_stream

    def run(strided):
        x = [t if strided else t.contiguous() for t in (q, k, v)]
        out = [torch.empty(s, dtype=d, device=dev()) for s, d in (
            ((B, NH, S, DV), torch.bfloat16), ((B, NH, DQK, DV), torch.float32), ((B, NH, DQK), torch.float32),
            ((B, NH), torch.float32))]
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev())
        rest = (i.data_ptr(), f.data_ptr(), None, None, None, *(t.data_ptr() for t in out), B, NH, S, DQK, DV, 64,
                DQK ** -0.5, 1e-6, 1, 1, 3, ws.data_ptr(), ws_bytes, st)
        if strided:
            strides = (ctypes.c_int64 * 9)(*[s for t in x for s in _strides(t)])
            rc = lib.xl_mlstm_chunkwise_fwd_strided(*(t.data_ptr() for t in x), strides, *rest)
        else:
            rc = lib.xl_mlstm_chunkwise_fwd(*(t.data_ptr() for t in x), *rest)
        _lib.check(rc, "strided" if strided else "contiguous")
        torch.cuda.synchronize()
        return out

    for a, b in zip(run(True), run(False)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("layout,copies", [("projection", False), ("packed", False), ("expanded", False),
                                           ("odd_rows", True), ("offset", True)])
def test_operator_reads_in_place(gpu_case, layout, copies):
    """The most memory a call holds: that of the contiguous call where it reads the views in place, three copies
    more where it cannot."""
    import xlstm_hip
    x = _views(2, 4, 1000, 128, 256, torch.bfloat16, layout, 3)

    def peak(x):
        torch.cuda.synchronize()
        base = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        xlstm_hip.mlstm_chunkwise(*x, algo="pipelined")
        torch.cuda.synchronize()
        return torch.cuda.max_memory_allocated() - base

    plain = tuple(t.contiguous() for t in x)
    peak(plain)
    more = peak(x) - peak(plain)
    assert more == (sum(t.numel() * 2 for t in plain[:3]) if copies else 0)


def test_strided_with_states_and_backend(gpu_case):
    import xlstm_hip
    q, k, v, i, f = _views(2, 4, 200, 128, 256, torch.bfloat16, "projection", 5)
    C, n, m = torch.randn(2, 4, 128, 256, device=dev()), torch.rand(2, 4, 128, device=dev()), torch.zeros(2, 4, 1, device=dev())
    backend = xlstm_hip.mLSTMBackend(xlstm_hip.mLSTMBackendConfig(mode="inference"))
    for states in ((None, None, None), (C, n, m)):
        a = backend(q, k, v, i, f, *states)
        b = backend(q.contiguous(), k.contiguous(), v.contiguous(), i, f, *states)
        z = (torch.zeros_like(C), torch.zeros_like(n), torch.zeros_like(m)) if states[0] is None else states
        c = backend(q, k, v, i, f, *z)  # no initial states: the zero state
        for x, y, w in zip((a[0], *a[1]), (b[0], *b[1]), (c[0], *c[1])):
            assert torch.equal(x, y) and torch.equal(x, w)


def test_strided_gradients(gpu_case):
    import xlstm_hip
    x = _views(1, 2, 128, 128, 256, torch.bfloat16, "projection", 7)
    grads = []
    for leaf in (x, tuple(t.contiguous() for t in x)):
        leaf = tuple(t.detach().requires_grad_(True) for t in leaf)
        h = xlstm_hip.mlstm_chunkwise(*leaf)
        grads.append(torch.autograd.grad(h, leaf, torch.ones_like(h)))
    for a, b in zip(*grads):
        assert torch.equal(a, b)
