"""Sizes at which gla's step of one token keeps its projections in launches of their own (no GPU: the rule)."""
import pytest

from nano_vllm_x_amd import ops


@pytest.mark.parametrize("n_seq,heads,dim,vdim,rank,one", [      # us of the one launch and of the four
    (48, 16, 64, 128, 16, True),          # 15.2 and 20.3
    (96, 8, 64, 128, 16, True),           # 13.9 and 19.1
    (128, 8, 64, 128, 16, False),         # 24.5 and 23.9
    (128, 16, 64, 128, 16, False),        # 46 and 39
    (256, 16, 64, 128, 16, False),        # 87 and 63
    (32, 32, 64, 128, 16, False),         # (4096 inputs) 31 and 27
    (96, 8, 64, 128, 32, True),           # 18.2 and 20.1
    (128, 8, 64, 128, 32, False),         # 31 and 25
    (96, 16, 64, 128, 4, True),           # 28.7 and 33.7
    (128, 16, 64, 128, 4, False),         # 39.1 and 38.5
    (128, 8, 128, 256, 16, True),         # 53 and 56
    (256, 8, 128, 256, 16, False),        # 102 and 101
    (128, 8, 64, 64, 16, False)])         # 19.0 and 18.2
def test_where_the_four_launches_are_the_faster(n_seq, heads, dim, vdim, rank, one):
    assert ops.gla_step_faster(n_seq, heads, dim, vdim, rank) is one
