"""What stands in a mixture's place in a Gibavik layer is called, with its hooks, whatever it hands on of the module that it wraps (no GPU: the calls only)."""
import pytest
import torch
from torch import nn

from nano_vllm_x_amd import gibavik
from nano_vllm_x_amd.layers import moe as moe_layers
from nano_vllm_x_amd.layers.moe import ExpertBank, TableMoE


class Halves(nn.Module):
    """Halves what the module inside gives; attributes of that module are its own."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def __getattr__(self, name):
        try:
            return super().__getattr__(name)
        except AttributeError:
            return getattr(super().__getattr__("inner"), name)

    def forward(self, *args, **kwargs):
        return 0.5 * self.inner(*args, **kwargs)


class Copies(nn.Module):
    """A module of its own with what a step's plan asks a mixture for."""

    def __init__(self, inner):
        super().__init__()
        self.top, self.experts, self.by_rows = inner.top, inner.experts, inner.by_rows
        self.register_buffer("table", inner.table)

    def forward(self, h, input_ids, decode_step=False, plan=None):
        return torch.full_like(h, 3.0)


def _forward(monkeypatch, change):
    cfg = gibavik.GibavikConfig.from_dict({
        "architecture": "Gibavik", "vocab": 16, "width": 64, "norm": {"eps": 1e-5}, "embedding": {"scale": 1.0}, "logit_softcap": 30.0,
        "layers": [{"type": "attention", "mixer": {"heads": 1, "kv_heads": 1, "dim": 64, "vdim": 64, "scale": 1.0}, "mlp": {"kind": "moe", "expert": {"ff": 64}, "router": {"experts": 4, "top": 2}}}]})
    m = gibavik.GibavikForCausalLM(cfg)
    layer, results = m.layers[0], []
    layer.mixer = type("Mixer", (nn.Module,), {"forward": lambda self, h, positions, md: h})()
    m.set_attention_metadata(type("Step", (), {"layout": type("Layout", (), {"qo_indptr": None})})())
    monkeypatch.setattr(gibavik.ops, "embed_scale", lambda ids, table, scale: (torch.zeros(len(ids), 64), torch.ones(len(ids), 64)))
    monkeypatch.setattr(gibavik.ops, "postnorm_residual", lambda x, y=None, **k: results.append(y) or y)
    monkeypatch.setattr(moe_layers.ops, "moe_expert_rows", lambda h, *a: torch.full_like(h, 2.0))
    monkeypatch.setattr(moe_layers.ops, "moe_expert_rows_postnorm", lambda *a: "in one launch")
    monkeypatch.setattr(TableMoE, "by_rows", lambda *a: True)
    seen = change(layer, monkeypatch)
    with torch.no_grad():
        out = m(torch.zeros(3, dtype=torch.int64), torch.arange(3))
    return out, results, seen


def test_a_mixture_as_it_was_built_ends_in_the_norms_launch(monkeypatch):
    assert _forward(monkeypatch, lambda layer, mp: None)[0] == "in one launch"


def test_a_wrapper_that_hands_look_ups_on_is_called_with_its_hooks(monkeypatch):
    def change(layer, mp):
        calls = []
        layer.mlp = Halves(layer.mlp)
        layer.mlp.register_forward_hook(lambda m, a, out: calls.append(out))
        return calls

    out, results, calls = _forward(monkeypatch, change)
    assert len(calls) == 1 and torch.equal(out, torch.ones(3, 64)) and torch.equal(results[-1], out)


def test_a_module_of_its_own_is_called(monkeypatch):
    out, results, _ = _forward(monkeypatch, lambda layer, mp: setattr(layer, "mlp", Copies(layer.mlp)))
    assert torch.equal(out, torch.full((3, 64), 3.0))


@pytest.mark.parametrize("where", ["instance", "class"])
def test_another_run_of_the_mixtures_own_is_called(monkeypatch, where):
    def change(layer, mp):
        def run(*a, **k):
            return torch.full((3, 64), 5.0)
        if where == "instance":
            layer.mlp.run = run
        else:
            mp.setattr(ExpertBank, "run", run)

    assert torch.equal(_forward(monkeypatch, change)[0], torch.full((3, 64), 5.0))
