"""The pipelined chunkwise kernel on q, k, v read in place from a projection's layout.

The strided call must be bit-equal to the call on contiguous copies (the same kernel, other addresses), over
head widths, ragged lengths, batches, the sequence split, f16, initial states, and views whose rows cannot be
read in place (odd row strides, an offset base, expanded rows), which take the copy."""

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
    return q / DQK ** 0.5 if layout == "plain_q" else q, k, v, i, f


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
