"""A block's element-wise kernels on the GPU: residual add + RMSNorm (with state copies), the SwiGLU product,
and the pair of gate projections in both output layouts.

Expected values are the modules' own torch composition evaluated in float64 with their 16-bit roundings.
Bar: one ulp of the output (an intermediate or the result may land on the other side of a rounding boundary
in float32), for silu(g) u also the half ulp that a flipped SiLU moves, relative to the product; the sum
x + r is exact to its rounding and must be bit-equal to torch's.  The gate pair must be bit-equal to the
single projection of the stacked weights (the same kernels)."""

import pytest
import torch

from helpers import dev

pytestmark = pytest.mark.gpu


def _ulp(x, dtype):
    mant = 7 if dtype == torch.bfloat16 else 10
    return torch.exp2(torch.floor(torch.log2(x.abs().clamp_min(2.0 ** -14))) - mant)


# D: one vector, a partial wave, one / two / four vectors per thread, past the registers (8192)
@pytest.mark.parametrize("M,D", [(1, 8), (3, 200), (8, 2048), (5, 4096), (2, 5504), (2, 8192), (3, 12296)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("residual", [False, True])
def test_add_rmsnorm(gpu_case, M, D, dtype, residual):
    from xlstm_hip.ops import add_rmsnorm_op, rms_norm_op
    g = torch.Generator().manual_seed(D + M)
    x, r = (torch.randn(M, D, generator=g).to(dtype).to(dev()) for _ in range(2))
    w = (1 + 0.1 * torch.randn(D, generator=g)).to(dtype).to(dev())
    if residual:
        src = [torch.randn(n, generator=g).to(dev()) for n in (1000, 7)]
        dst = [torch.zeros_like(t) for t in src]
        s, y = add_rmsnorm_op(x, r, w, 1e-6, src, dst)
        assert torch.equal(s, x + r)
        assert all(torch.equal(a, b) for a, b in zip(src, dst))
    else:
        s, y = x, rms_norm_op(x, w, 1e-6)
    sd = s.double()
    want = sd * torch.rsqrt((sd * sd).mean(-1, keepdim=True) + 1e-6) * w.double()
    assert float(((y.double() - want).abs() - _ulp(want, dtype)).max()) <= 0


def test_longest_state_copy(gpu_case):
    """A copy of 2^31 - 1 values, the most an int names, by a grid whose stride takes the index past it: whole, and
    nothing beside it."""
    from xlstm_hip.ops import add_rmsnorm_op
    n = 2 ** 31 - 1
    src = torch.full((n,), 2.0, device=dev())
    src[-1] = 3.0
    whole = torch.zeros(n + 64, device=dev())
    x, w = torch.ones(4096, 8, dtype=torch.bfloat16, device=dev()), torch.ones(8, dtype=torch.bfloat16, device=dev())
    add_rmsnorm_op(x, x, w, 1e-6, [src], [whole[:n]])
    assert float(whole[n - 1]) == 3.0 and not whole[n:].any()
    assert float(whole[:n - 1].min()) == float(whole[:n - 1].max()) == 2.0


@pytest.mark.parametrize("shape", [(1, 8), (3, 5504), (4100, 2752)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_mul(gpu_case, shape, dtype):
    from xlstm_hip.ops import silu_mul_op
    g = torch.Generator().manual_seed(shape[0])
    a, b = ((3 * torch.randn(shape, generator=g)).to(dtype) for _ in range(2))
    y = silu_mul_op(a.to(dev()), b.to(dev())).double().cpu()
    sl = (a.double() * torch.sigmoid(a.double())).to(dtype).double()
    want = sl * b.double()
    bar = _ulp(want, dtype) + _ulp(sl, dtype) * b.double().abs()
    assert float(((y - want).abs() - bar).max()) <= 0


# row form (D 2048, G 8; one slice set per G) and tile form (D 4096; D no multiple of 512), ragged rows,
# uneven pairs, a missing bias
@pytest.mark.parametrize("B,S,D,G1,G2", [(1, 1, 2048, 4, 4), (3, 37, 2048, 4, 4), (2, 50, 4096, 8, 8), (1, 17, 200, 3, 5),
                                         (2, 16, 512, 24, 40), (1, 33, 1024, 1, 2)])
@pytest.mark.parametrize("heads_first", [False, True])
@pytest.mark.parametrize("cap_in_dtype", [False, True])
def test_gate_pair(gpu_case, B, S, D, G1, G2, heads_first, cap_in_dtype):
    from xlstm_hip.mlstm_layers import gate_pair_softcap, gate_proj_softcap, stacked_linears
    torch.manual_seed(D + S)
    l1, l2 = torch.nn.Linear(D, G1), torch.nn.Linear(D, G2, bias=G1 != 3)
    l1, l2 = (m.to(torch.bfloat16).to(dev()) for m in (l1, l2))
    x = torch.randn(B, S, D).to(torch.bfloat16).to(dev())
    with torch.no_grad():
        y1, y2 = gate_pair_softcap(x, l1, l2, 15.0, cap_in_dtype, heads_first)
        y = gate_proj_softcap(x, *stacked_linears(l1, l2), 15.0, cap_in_dtype)
    w1, w2 = y[..., :G1], y[..., G1:]
    if heads_first:
        w1, w2 = w1.permute(0, 2, 1), w2.permute(0, 2, 1)
    assert y1.is_contiguous() and torch.equal(y1, w1)
    assert y2.is_contiguous() and torch.equal(y2, w2)


def test_stack_decode_matches_modules(gpu_case):
    """decode_step with the one-pass kernels against the same blocks run through torch's own norms and
    SwiGLU: the last bit of a norm may move and travels through the blocks, so to 1 % of the logits' scale."""
    import xlstm_hip.stack as st
    cfg = st.StackConfig("small", d_model=512, num_blocks=4, mlstm_heads=4, slstm_every=4, vocab=1000)
    model = st.xLSTMStack.random(cfg, dev(), seed=3)
    tok = torch.arange(3, device=dev())
    prompt = torch.arange(60, device=dev()).view(3, 20)
    out = []
    for one_pass in (st._one_pass, lambda *a: False):
        keep, st._one_pass = st._one_pass, one_pass
        try:
            _, states = model.prefill(prompt)
            out.append(torch.stack([model.decode_step(tok + i, states) for i in range(3)]))
        finally:
            st._one_pass = keep
    a, b = (t.double() for t in out)
    assert float((a - b).abs().max()) <= 1e-2 * float(b.abs().max())
