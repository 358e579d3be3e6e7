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
