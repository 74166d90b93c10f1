"""What keeps a mixture's sums out of the norm's launch: whatever hangs on the module's call."""
import pytest
import torch

from nano_vllm_x_amd.layers.moe import TableMoE
from nano_vllm_x_amd import ops


@pytest.mark.parametrize("what", ["nothing", "hook", "pre-hook", "own forward", "class", "patched", "mode", "weight"])
def test_the_call_is_made_where_something_hangs_on_it(what, monkeypatch):
    m = (type("Other", (TableMoE,), {}) if what == "class" else TableMoE)(64, 4, 2, 64, 10)
    monkeypatch.setattr(TableMoE, "by_rows", lambda *a: True)
    monkeypatch.setattr(ops, "moe_expert_rows_postnorm", lambda *a: "made")
    if what == "hook":
        m.register_forward_hook(lambda *a: None)
    elif what == "pre-hook":
        m.register_forward_pre_hook(lambda *a: None)
    elif what == "own forward":
        m.forward = lambda *a, **k: None
    elif what == "patched":
        monkeypatch.setattr(TableMoE, "forward", lambda *a, **k: None)
    elif what == "weight":
        m.w_gu = type("P", (torch.nn.Parameter,), {})(m.w_gu.data)
    h = torch.zeros(3, 64)
    with torch.overrides.BaseTorchFunctionMode() if what == "mode" else torch.no_grad():
        got = m.into_stream(h, False, {"idx": None, "wts": None, "order": None}, h, torch.ones(1), 1e-5)
    assert (got == "made") if what == "nothing" else (got is None)
