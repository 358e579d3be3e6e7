"""The backward's fused path (bf16, DV 256 / 512) where its launches change form: n and m in blocks of 64 chunks
(more than 64, one past a block), both row widths of the paired scans (64 rows up to 128 workgroups of 128, 128
beyond), and workgroup counts that are no multiple of 8 (the XCD grouping).  Bars of test_gpu_chunkwise_bwd.py."""

import pytest
import torch

from test_gpu_chunkwise_bwd import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,NH,S,DQK,DV", [(1, 1, 64 * 65, 128, 256),    # one chunk past a block of 64
                                           (1, 2, 64 * 64, 64, 256),     # exactly a block
                                           (3, 6, 64, 128, 512),         # 288 workgroups of 128 rows
                                           (1, 8, 128, 128, 512),        # 128: the last that takes 64 rows
                                           (1, 9, 128, 128, 512),        # 144: the first that takes 128
                                           (1, 9, 192, 256, 512),        # 288, two row slices a state
                                           (1, 1, 128, 128, 256)])
@pytest.mark.parametrize("states", [False, True])
def test_forms(gpu_case, B, NH, S, DQK, DV, states):
    _run(B, NH, S, DQK, DV, 64, torch.bfloat16, states, states, seed=S + DQK + B)


@pytest.mark.parametrize("B,NH,S,DQK,DV", [(1, 2, 192, 256, 128), (1, 8, 64, 128, 1024), (1, 9, 64, 128, 1024),
                                           (1, 24, 64, 128, 1024), (1, 25, 64, 128, 1024)])
def test_float32_row_slices(gpu_case, B, NH, S, DQK, DV):
    """The float32 scans with 64 rows a workgroup (up to 384 workgroups of 128 rows: 4 slices of a state, 128, 144,
    exactly 384) and 128 (400), forward and backward."""
    _run(B, NH, S, DQK, DV, 64, torch.float32, True, True, seed=DV)


@pytest.mark.parametrize("DQK", [64, 128, 256])
@pytest.mark.parametrize("DV", [256, 512])
@pytest.mark.parametrize("S", [64, 1024 + 64])
def test_gate_partials(gpu_case, DQK, DV, S):
    """The gate pass at every count of partials that the fused path has, in one 1024-token segment and two."""
    _run(1, 2, S, DQK, DV, 64, torch.bfloat16, False, True, seed=DQK + DV)
