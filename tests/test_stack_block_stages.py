"""Which calls a block's one-pass kernels take (fake GPU tensors, no GPU): what they cannot do runs as torch's own
add, norm, SiLU and copies, as it did without them."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

D = 64
BF = torch.bfloat16


def _norm():
    from xlstm_hip.stack import _RMSNorm
    norm = _RMSNorm(D, 1e-6)
    norm.weight = torch.nn.Parameter(torch.ones(D, device="cuda", dtype=BF), requires_grad=False)
    return norm


def _x(*shape, dtype=BF):
    return torch.randn(*(shape or (2, 3, D)), device="cuda", dtype=dtype)


@pytest.fixture
def seen(monkeypatch):
    """The one-pass operators called: the name, and the state copies given to add_rmsnorm."""
    import xlstm_hip.stack as st
    calls = []
    for name in ("add_rmsnorm_op", "rms_norm_op", "silu_mul_op"):
        op = getattr(st, name)

        def call(*a, _op=op, _n=name):
            calls.append(_n + str(len(a[4])) if len(a) > 4 else _n)
            return _op(*a)

        monkeypatch.setattr(st, name, call)
    return calls


def test_taken(seen):
    from xlstm_hip.stack import _add_norm
    with FakeTensorMode():
        src, dst = torch.randn(2, 3, device="cuda"), torch.zeros(2, 3, device="cuda")
        s, y = _add_norm(_x(), _x(), _norm(), ((src, dst),))
        assert s.shape == y.shape == (2, 3, D) and dst._version == 1
        _add_norm(_x(), None, _norm())
    assert seen == ["add_rmsnorm_op1", "rms_norm_op"]


# the residual alone requires a gradient, has another dtype, broadcasts
@pytest.mark.parametrize("r", ["grad", "dtype", "broadcast"])
def test_residual_the_kernel_cannot_add(seen, r):
    from xlstm_hip.stack import _add_norm
    with FakeTensorMode():
        res = {"grad": lambda: _x().requires_grad_(True), "dtype": lambda: _x(dtype=torch.float32),
               "broadcast": lambda: _x(D)}[r]()
        s, y = _add_norm(_x(), res, _norm())
        assert s.shape == y.shape == (2, 3, D) and s.dtype == (torch.float32 if r == "dtype" else BF)
        assert s.requires_grad == y.requires_grad == (r == "grad")
        if r == "grad":
            assert type(s.grad_fn).__name__ == "AddBackward0"
    assert "add_rmsnorm_op0" not in seen


@pytest.mark.parametrize("dst", ["strided", "half", "broadcast", "three"])
def test_state_copies_the_kernel_cannot_make(seen, dst):
    from xlstm_hip.stack import _add_norm
    with FakeTensorMode():
        src = torch.randn(4, 6, device="cuda")
        to = {"strided": torch.zeros(6, 4, device="cuda").t(), "half": torch.zeros(4, 6, device="cuda", dtype=BF),
              "broadcast": torch.zeros(5, 4, 6, device="cuda"), "three": torch.zeros(4, 6, device="cuda")}[dst]
        copies = ((src, to),) * (3 if dst == "three" else 1)
        _add_norm(_x(), _x(), _norm(), copies)
        assert to._version == len(copies)
    assert seen == ["add_rmsnorm_op0"]


def test_transforms_take_torchs_own_stages(seen):
    import torch.autograd.forward_ad as fa
    from xlstm_hip.stack import _one_pass
    with FakeTensorMode():
        x, norm = _x(), _norm()
        assert _one_pass(x, norm.weight)
        with fa.dual_level():  # torch's norm has a forward-mode derivative, the kernel has none
            assert not _one_pass(x, norm.weight)
        assert torch.vmap(norm)(x).shape == (2, 3, D)
    assert seen == []
