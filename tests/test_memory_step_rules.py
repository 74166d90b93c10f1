"""Sizes at which the steps of one token of gla and mlstm keep their projections in launches of their own (no GPU: the rules)."""
import types

import pytest
import torch

from nano_vllm_x_amd import ops
from nano_vllm_x_amd.layers import recurrent


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


def test_rows_of_another_format_and_inputs_that_no_projection_takes_keep_the_separate_launches():
    """A replaced projection may give its rows in a format of its own, which the separate launches read; more than 12288 inputs they refuse."""
    lay = types.SimpleNamespace(qo_indptr=None, n_tok=3)
    mem, w = torch.zeros(3, 2, 64, 64), lambda r, k=64: torch.zeros(r, k)
    h, x = torch.zeros(3, 64).bfloat16(), torch.zeros(3, 512)
    for w1, w2 in ((w(4), None), (w(16), w(128, 16))):
        assert ops.memory_step_fits(lay, h, mem, w1, w2, x=x.bfloat16()) and ops.memory_step_fits(lay, x[:, :64], mem, w1, w2, x=x)
        assert not ops.memory_step_fits(lay, h, mem, w1, w2, x=x) and not ops.memory_step_fits(lay, h, mem, w1, w2, x=x.half())
    assert ops.memory_step_fits(lay, torch.zeros(3, 12288), mem, w(4, 12288), x=x) and not ops.memory_step_fits(lay, torch.zeros(3, 12292), mem, w(4, 12292), x=x)


def test_the_modules_ask_with_their_rows(monkeypatch):
    asked = []
    monkeypatch.setattr(ops, "memory_step_fits", lambda layout, h, *a, x=None: asked.append((h.dtype, x.dtype)) or False)
    for name in ("skinny_proj", "mlstm_scan", "gla_scan"):
        monkeypatch.setattr(ops, name, lambda *a, **k: None)
    monkeypatch.setattr(ops, "head_norm_gate", lambda *a, gate, **k: gate)
    md = types.SimpleNamespace(layout=None, cache=types.SimpleNamespace(state=lambda key: None))
    for m in (recurrent.MLSTM(64, 1, 64, 64, 15.0, 1e-5, "s"), recurrent.GatedLinearAttention(64, 1, 64, 64, 16.0, 16, 1e-5, "s")):
        m.qkvg_proj.forward = lambda h: torch.zeros(len(h), 256)
        m.o_proj.forward = lambda y: y
        assert m(torch.zeros(3, 64).bfloat16(), md).dtype == torch.float32
    assert asked == [(torch.bfloat16, torch.float32)] * 2
