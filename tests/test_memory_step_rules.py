"""Sizes at which the steps of one token of gla and mlstm keep their projections in launches of their own (no GPU: the rules)."""
import pytest

from nano_vllm_x_amd import ops


@pytest.mark.parametrize("n_seq,heads,dim,vdim,rank,one", [      # us of the one launch and of the four
    (48, 16, 64, 128, 16, True),          # 15.2 and 20.5
    (96, 8, 64, 128, 16, True),           # 13.8 and 19.0
    (128, 8, 64, 128, 16, False),         # 24.9 and 23.9
    (128, 16, 64, 128, 16, False),        # 45.5 and 37.2
    (256, 16, 64, 128, 16, False),        # 86 and 57
    (32, 32, 64, 128, 16, False),         # (4096 inputs) 31 and 27
    (96, 8, 64, 128, 32, True),           # 18.0 and 20.0
    (128, 8, 64, 128, 32, False),         # 31 and 25
    (96, 16, 64, 128, 4, True),           # 28.3 and 31.8
    (128, 16, 64, 128, 4, False),         # 39.8 and 36.9
    (128, 8, 128, 256, 16, True),         # 53 and 55
    (256, 8, 128, 256, 16, False),        # 102 and 103
    (128, 8, 64, 64, 16, False)])         # 19.0 and 18.2
def test_where_the_four_launches_are_the_faster(n_seq, heads, dim, vdim, rank, one):
    assert ops.gla_step_faster(n_seq, heads, dim, vdim, rank) is one


@pytest.mark.parametrize("n_seq,heads,dim,vdim,one", [      # us of the one launch and of the three
    (128, 16, 64, 128, True),             # 31.0 and 34.4
    (256, 8, 64, 128, True),              # 30.0 and 33.2
    (192, 16, 64, 128, False),            # 45.0 and 44.4
    (256, 16, 64, 128, False),            # 59.0 and 54.3
    (256, 16, 64, 64, False),             # 42.4 and 36.1
    (256, 16, 128, 128, True),            # 95.6 and 98.9
    (256, 16, 256, 256, True)])           # 419 and 435
def test_where_the_three_launches_of_mlstm_are_the_faster(n_seq, heads, dim, vdim, one):
    assert ops.mlstm_step_faster(n_seq, heads, dim, vdim) is one
