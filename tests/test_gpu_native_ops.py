"""The native operator kernels under torch's own machinery: autograd (hooks on saved tensors, checkpointing,
double backward), tracing, in-place version counters, threads and streams, and what is refused."""

import threading

import pytest
import torch

from helpers import dev

pytestmark = pytest.mark.gpu


def _x(S=128, seed=0, dtype=torch.bfloat16, grad=False):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(1, 2, S, d, generator=g) for d in (128, 128, 256))
    i, f = torch.randn(1, 2, S, generator=g), torch.randn(1, 2, S, generator=g) + 3
    return tuple(t.to(dtype).to(dev()).requires_grad_(grad) for t in (q / 11, k, v, i, f))


def _grads(fn, x):
    h = fn(*x)
    return (h.detach(),) + torch.autograd.grad(h, x, torch.ones_like(h))


def _equal(a, b):
    return all(torch.equal(s, t) for s, t in zip(a, b))


@pytest.mark.parametrize("S", [128, 100])
def test_autograd_machinery(gpu_case, S):
    import xlstm_hip
    from torch.utils.checkpoint import checkpoint
    fn = lambda *x: xlstm_hip.mlstm_chunkwise(*x, algo="pipelined")  # noqa: E731
    x = _x(S, grad=True)
    want = _grads(fn, x)
    with torch.autograd.graph.save_on_cpu():
        assert _equal(_grads(fn, x), want)
    assert _equal(_grads(lambda *t: checkpoint(fn, *t, use_reentrant=False), x), want)
    with torch.no_grad():
        assert torch.equal(fn(*x), want[0]) and not fn(*x).requires_grad
    # some inputs only
    h = fn(x[0], *(t.detach() for t in x[1:]))
    assert torch.equal(torch.autograd.grad(h, x[0], torch.ones_like(h))[0], want[1])


def test_compiled(gpu_case):
    import xlstm_hip

    def fn(q, k, v, i, f):
        return xlstm_hip.mlstm_chunkwise(q * 1.0, k, v, i, f)

    x = _x(grad=True)
    got = _grads(torch.compile(fn, backend="aot_eager", fullgraph=True), x)
    assert _equal(got, _grads(fn, x))


def test_compiled_once_for_every_length(gpu_case):
    import xlstm_hip
    from torch._dynamo.testing import CompileCounterWithBackend
    count = CompileCounterWithBackend("aot_eager")

    def fn(q, k, v, i, f):
        return xlstm_hip.mlstm_chunkwise(q * 1.0, k, v, i, f)

    compiled = torch.compile(fn, backend=count, fullgraph=True, dynamic=True)
    for S in (192, 320, 448):  # (128 and 256 are head widths, which tracing would tie the length to)
        x = _x(S, seed=S, grad=True)
        assert _equal(_grads(compiled, x), _grads(fn, x))
    assert count.frame_count == 1


def test_refused(gpu_case):
    import xlstm_hip
    x = torch.randn(8, 16, device=dev(), requires_grad=True)
    with pytest.raises(RuntimeError):
        xlstm_hip.soft_cap(x, 15.0).sum().backward()  # forward-only
    q = _x(grad=True)
    h = xlstm_hip.mlstm_chunkwise(*q)
    g = torch.autograd.grad(h, q[0], torch.ones_like(h), create_graph=True)[0]
    with pytest.raises(RuntimeError):
        g.sum().backward()  # no second derivative
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: xlstm_hip.mlstm_chunkwise(t, *(u.detach() for u in q[1:])).sum())(q[0].detach())
    with pytest.raises(RuntimeError, match="no CPU path"):
        xlstm_hip.soft_cap(x.detach().cpu(), 15.0)
    with pytest.raises(RuntimeError, match="no CPU path"):
        xlstm_hip.mlstm_chunkwise(q[0].detach(), q[1].detach().cpu(), *(t.detach() for t in q[2:]))
    with pytest.raises(ValueError, match="share a dtype"):
        xlstm_hip.mlstm_chunkwise(q[0].detach(), q[1].detach().float(), *(t.detach() for t in q[2:]))
    with pytest.raises(ValueError, match="unsupported dtype"):
        xlstm_hip.soft_cap(torch.arange(8, device=dev()), 15.0)
    with pytest.raises(AssertionError, match="not divisible"):
        xlstm_hip.mlstm_chunkwise(*_x(100))


def test_in_place_version(gpu_case):
    import xlstm_hip
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(1, 2, d, generator=g).to(dev()) for d in (64, 64, 128))
    i, f, m = (torch.randn(1, 2, 1, generator=g).to(dev()) for _ in range(3))
    C, n = torch.randn(1, 2, 64, 128, generator=g).to(dev()), torch.rand(1, 2, 64, generator=g).to(dev())
    before = C._version
    xlstm_hip.mlstm_recurrent_step_(q, k, v, i, f, C, n, m)
    assert C._version > before


def test_threads_and_streams(gpu_case):
    """Four threads, each on its own stream with its own inputs, against the same calls in turn."""
    import xlstm_hip
    xs = [_x(64 * (8 + s), seed=s) for s in range(4)]
    want = [xlstm_hip.mlstm_chunkwise(*x, return_last_states=True) for x in xs]
    torch.cuda.synchronize()
    got = [None] * 4

    def work(s):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for _ in range(5):
                got[s] = xlstm_hip.mlstm_chunkwise(*xs[s], return_last_states=True)
        st.synchronize()

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    for a, b in zip(got, want):
        assert torch.equal(a[0], b[0]) and _equal(a[1], b[1])
