"""The single-pass forward's workspace (no GPU): each schedule asks for its own per-segment states and no more."""

import pytest
import torch


def _segments(B, NH, S, DQK, DV, algo):
    """The workspace past the gate prep, and the bytes of one segment's states (C, n, m and, in the pipelined
    schedule, the total log forget gate)."""
    from xlstm_hip.ops import chunkwise_workspace_bytes
    total = chunkwise_workspace_bytes(B, NH, S, DQK, DV, 64, torch.bfloat16, algo=algo)
    prep = -(-B * NH * -(-S // 64) * 1280 // 256) * 256
    return total - prep, B * NH * (DQK * DV + DQK + (2 if algo == "pipelined" else 1)) * 4


# one column tile (15 end states at most), the 7B head's prompt, no split
@pytest.mark.parametrize("B,NH,S,DQK,DV,most", [(1, 1, 64 * 130, 128, 64, 15), (1, 8, 2011, 256, 512, 4),
                                                (1, 2, 2048, 256, 128, 15), (4, 8, 8192, 256, 512, 0)])
def test_pipelined_workspace_holds_end_states_only(B, NH, S, DQK, DV, most):
    states, one = _segments(B, NH, S, DQK, DV, "pipelined")
    assert states <= most * one + 256
    fused, one = _segments(B, NH, S, DQK, DV, "fused")
    assert fused <= 2 * 15 * one + 512


# Calls timed split and unsplit: one launch where the second one costs more than it saves (6 to 12 chunks), the
# split where it was the faster (the 7B head's prompt among them)
@pytest.mark.parametrize("B,NH,NC,DQK,DV,split", [(1, 4, 6, 256, 512, False), (1, 4, 7, 256, 512, False),
                                                  (1, 8, 7, 256, 512, False), (2, 8, 10, 256, 512, False),
                                                  (2, 8, 12, 256, 512, False), (1, 8, 6, 192, 384, False),
                                                  (1, 2, 6, 32, 64, False), (2, 8, 6, 64, 128, False),
                                                  (1, 8, 6, 96, 192, False), (1, 8, 7, 96, 192, True),
                                                  (1, 2, 6, 128, 256, True), (1, 8, 7, 128, 256, True),
                                                  (1, 8, 9, 256, 512, True), (1, 8, 8, 64, 128, True),
                                                  (1, 8, 32, 256, 512, True), (2, 8, 64, 256, 512, True)])
def test_split_where_it_is_the_faster(B, NH, NC, DQK, DV, split):
    states, _ = _segments(B, NH, 64 * NC, DQK, DV, "pipelined")
    assert (states > 0) == split


# the fewest chunks that split, 8 heads: one fewer runs in one launch
@pytest.mark.parametrize("DQK,DV,first", [(32, 64, 7), (64, 128, 8), (96, 192, 7), (128, 256, 6), (192, 384, 8),
                                          (256, 512, 8)])
def test_first_split(DQK, DV, first):
    assert [_segments(1, 8, 64 * NC, DQK, DV, "pipelined")[0] > 0 for NC in range(1, 20)] == [
        NC >= first for NC in range(1, 20)]
