"""The operators under tracing and in-place bookkeeping, on fake tensors (no GPU): a training step traced with
symbolic shapes keeps its sizes symbolic."""

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx


def _trace(S, algo, states):
    import xlstm_hip
    x = [torch.randn(2, 3, S, 64), torch.randn(2, 3, S, 64), torch.randn(2, 3, S, 128), torch.randn(2, 3, S),
         torch.randn(2, 3, S)]
    if states:
        x += [torch.randn(2, 3, 64, 128), torch.rand(2, 3, 64), torch.randn(2, 3, 1)]

    def step(*x):
        x = [t.detach().requires_grad_(True) for t in x]
        h, (C, _, _) = xlstm_hip.mlstm_chunkwise(*x, algo=algo, return_last_states=True)
        return torch.autograd.grad(h.sum() + C.sum(), x)

    return make_fx(step, tracing_mode="symbolic")(*x)


# whole chunks, with initial states, and a ragged sequence (padded in the backward)
@pytest.mark.parametrize("S,algo,states", [(128, "auto", False), (128, "auto", True), (100, "pipelined", False)])
def test_training_step_traces_with_symbolic_sizes(S, algo, states):
    gm = _trace(S, algo, states)
    called = [str(n.target) for n in gm.graph.nodes if "xlstm_hip" in str(n.target)]
    assert called == ["xlstm_hip.mlstm_chunkwise.default", "xlstm_hip.mlstm_chunkwise_bwd.default"]
    q = next(n for n in gm.graph.nodes if n.op == "placeholder").meta["val"]
    assert all(not d.node.expr.is_number for d in q.shape), f"sizes fixed to the traced ones: {q.shape}"


def _step_inputs(leaf):
    q, k, v = (torch.randn(1, 2, d, device="cuda") for d in (64, 64, 128))
    i, f, m = (torch.randn(1, 2, 1, device="cuda") for _ in range(3))
    return (q, k, v, i, f), torch.randn(1, 2, 64, 128, device="cuda", requires_grad=leaf), torch.rand(1, 2, 64, device="cuda"), m


def test_in_place_ops_move_version_counters_under_fake_tensors():
    import xlstm_hip
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        x, C, n, m = _step_inputs(False)
        before = C._version
        xlstm_hip.mlstm_recurrent_step_(*x, C, n, m)
        assert C._version == before + 1
        a, w = torch.randn(2, 16, device="cuda", dtype=torch.bfloat16), torch.ones(16, device="cuda", dtype=torch.bfloat16)
        src, dst = torch.randn(4, device="cuda"), torch.zeros(4, device="cuda")
        torch.ops.xlstm_hip.add_rmsnorm(a, a, w, 1e-6, [src], [dst])
        assert dst._version == 1 and src._version == 0


@pytest.mark.parametrize("where", ["leaf C", "computed C", "q"])
def test_in_place_step_where_a_gradient_is_wanted(where):
    """C may require a gradient, as a leaf too: it is updated outside autograd (its own history stays), and
    a backward through the outputs raises."""
    import xlstm_hip
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        x, C, n, m = _step_inputs(where != "q")
        if where == "q":
            x[0].requires_grad_(True)
        elif where == "computed C":
            C = C * 1.0
        history = C.grad_fn
        h, (_, n1, m1) = xlstm_hip.mlstm_recurrent_step_(*x, C, n, m)
        assert C.grad_fn is history and C._version == 1
        assert h.grad_fn is not None and n1.grad_fn is not None and m1.grad_fn is not None
        with pytest.raises(RuntimeError):
            n1.grad_fn(None, torch.ones_like(n1), None)
    with torch.no_grad(), FakeTensorMode():
        x, C, n, m = _step_inputs(True)
        h, _ = xlstm_hip.mlstm_recurrent_step_(*x, C, n, m)
        assert not h.requires_grad


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_backend_traces_with_symbolic_sizes(dtype):
    """The any-length wrapper looks up whether the head's widths run in one call: they are taken as numbers, the
    length is not."""
    import xlstm_hip
    backend = xlstm_hip.mLSTMBackend(xlstm_hip.mLSTMBackendConfig(mode="inference"))
    x = [t.to(dtype) for t in (torch.randn(2, 3, 100, 64), torch.randn(2, 3, 100, 64), torch.randn(2, 3, 100, 128),
                               torch.randn(2, 3, 100), torch.randn(2, 3, 100))]
    gm = make_fx(lambda *x: backend(*x), tracing_mode="symbolic")(*x)
    called = [str(n.target) for n in gm.graph.nodes if "xlstm_hip" in str(n.target)]
    assert called.count("xlstm_hip.mlstm_chunkwise.default") == (1 if dtype == torch.bfloat16 else 2)
    q = next(n for n in gm.graph.nodes if n.op == "placeholder").meta["val"]
    assert all(not d.node.expr.is_number for d in q.shape[:3])
