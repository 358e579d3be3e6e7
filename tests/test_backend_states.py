"""Initial states of the any-length wrapper in the single-pass call (no GPU): none given, none passed; some given, the
others zero; all given, passed as they are."""

import pytest
import torch


@pytest.mark.parametrize("given", ["", "c", "n", "m", "cm", "cnm"])
def test_initial_states_of_the_single_pass_call(monkeypatch, given):
    from xlstm_hip import backend
    B, NH, S, DQK, DV = 2, 3, 100, 64, 128
    full = {"c": torch.randn(B, NH, DQK, DV), "n": torch.rand(B, NH, DQK), "m": torch.randn(B, NH, 1)}
    calls = []

    def kernel(**kw):
        calls.append(kw)
        return "h", ("C", "n", "m")

    monkeypatch.setattr(backend, "mlstm_chunkwise__native_autograd", kernel)
    monkeypatch.setattr(backend, "_fused_takes_any_length", lambda q, k, v: True)
    q, k, v = torch.randn(B, NH, S, DQK), torch.randn(B, NH, S, DQK), torch.randn(B, NH, S, DV)
    out = backend.wrap_chunkwise__arbitrary_sequence_length(
        kernel, None, None, q, k, v, q[..., 0], q[..., 0], **{f"{s}_initial": full[s] for s in given})
    assert out == ("h", ("C", "n", "m")) and len(calls) == 1
    kw = calls[0]
    assert kw["q"] is q and kw["chunk_size"] == 64 and kw["algo"] == "pipelined"
    for s in "cnm":
        t = kw[f"{s}_initial"]
        if not given:
            assert t is None
        elif s in given:
            assert t is full[s]
        else:
            assert t.shape == full[s].shape and t.dtype == torch.float32 and not t.any()
