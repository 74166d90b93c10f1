"""The attention of prompts reads a plan exactly where the wrapper makes one (no GPU: which launches are asked for)."""
import pytest
import torch

from nano_vllm_x_amd import _lib, ops
from nano_vllm_x_amd.layers.attention import PagedPrefillWrapper


def test_the_limit_is_the_kernels():
    assert ops.prefill_planless() == _lib.load().nvx_internal_prefill_planless() > 0


@pytest.mark.parametrize("more", [-1, 0, 1])
def test_a_plan_is_made_for_more_sequences_only(monkeypatch, more):
    made, n = [], ops.prefill_planless() + more
    monkeypatch.setattr(ops, "prefill_plan_ws", lambda batch, device: torch.zeros(3 * (batch + 2), dtype=torch.int32))
    monkeypatch.setattr(torch.ops, "nvx", type("Ops", (), {"prefill_plan": staticmethod(lambda *a: made.append(a))}))
    w = PagedPrefillWrapper()
    w.plan(torch.arange(n + 1, dtype=torch.int32), torch.arange(n + 1, dtype=torch.int32), torch.arange(n, dtype=torch.int32), None, 2, 1, 128)
    assert len(made) == (more > 0)
