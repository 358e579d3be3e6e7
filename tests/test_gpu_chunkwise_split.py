"""The pipelined kernel's split of the sequence into segments, at its edges: the fewest chunks that split, a
ragged and a one-chunk last segment, many segments (few heads: 15, composed four at a time), narrow heads, an
initial state, and input gates of -inf in a whole segment.  Against the float32 oracle at the 16-bit bar; each case
names its number of segments a launch, which the workspace shows, so that none passes unsplit."""

import pytest
import torch

from helpers import assert_parity, dev
from oracle import mlstm as om
from test_chunkwise_workspace import _segments

pytestmark = pytest.mark.gpu


# NC 6 .. 130 at 1 .. 128 column tiles of the batch
@pytest.mark.parametrize("B,NH,S,DQK,DV,w", [(1, 8, 64 * 9, 256, 512, 4), (1, 8, 64 * 11 + 1, 128, 256, 6),
                                             (1, 1, 64 * 33, 64, 64, 11), (1, 1, 64 * 130 - 7, 32, 64, 14),
                                             (2, 8, 64 * 8 + 40, 96, 192, 4), (1, 3, 64 * 23, 192, 128, 11),
                                             (1, 2, 64 * 16, 256, 64, 8), (2, 8, 64 * 26 + 63, 128, 512, 2),
                                             (1, 5, 64 * 6, 128, 64, 5)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("with_state", [False, True])
def test_split_edges(gpu_case, B, NH, S, DQK, DV, w, dtype, with_state):
    import xlstm_hip
    states, one = _segments(B, NH, S, DQK, DV, "pipelined")
    assert states // one == w
    g = torch.Generator().manual_seed(S + DV)
    q = torch.randn(B, NH, S, DQK, generator=g) / DQK ** 0.5
    k, v = torch.randn(B, NH, S, DQK, generator=g), torch.randn(B, NH, S, DV, generator=g)
    i, f = torch.randn(B, NH, S, generator=g), torch.randn(B, NH, S, generator=g) + 3
    x = tuple(t.to(dtype) for t in (q, k, v, i, f))
    st = (0.1 * torch.randn(B, NH, DQK, DV, generator=g), torch.rand(B, NH, DQK, generator=g),
          torch.randn(B, NH, 1, generator=g)) if with_state else (None, None, None)
    h, last = xlstm_hip.mlstm_chunkwise(*(t.to(dev()) for t in x), *(None if t is None else t.to(dev()) for t in st),
                                        return_last_states=True, algo="pipelined")
    hr, lr = om.mlstm_recurrent_sequence(*(t.float() for t in x), *st, return_last_states=True)
    for got, want, name in zip((h, *last), (hr, *lr), "hCnm"):
        assert_parity(got, want, dtype, name)


def test_split_closed_input_gates(gpu_case):
    """Input gates of -inf over more than one segment: nothing enters, the state only decays."""
    import xlstm_hip
    B, NH, S, DQK, DV = 1, 8, 64 * 24, 128, 256
    assert _segments(B, NH, S, DQK, DV, "pipelined")[0] > 0
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(B, NH, S, d, generator=g).to(torch.bfloat16) for d in (DQK, DQK, DV))
    i, f = torch.randn(B, NH, S, generator=g), torch.randn(B, NH, S, generator=g) + 6
    i[:, :, 64 * 8:] = -float("inf")
    h, last = xlstm_hip.mlstm_chunkwise(*(t.to(dev()) for t in (q, k, v, i, f)), return_last_states=True, algo="pipelined")
    hr, lr = om.mlstm_recurrent_sequence(*(t.float() for t in (q, k, v, i, f)), return_last_states=True)
    for got, want, name in zip((h, *last), (hr, *lr), "hCnm"):
        assert_parity(got, want, torch.bfloat16, name)
