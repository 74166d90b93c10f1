"""Which Qwen3 decode steps may carry their norms on their products, modules not called: those of a stack as it was built (no GPU: only the choice)."""
import pytest
import torch
from torch import nn

import test_plain_calls as plain_calls
from nano_vllm_x_amd import ops, qwen3
from nano_vllm_x_amd.core.common import ForwardMode
from nano_vllm_x_amd.layers.attention import AttentionMetadata, PagedDecodeWrapper, PagedPrefillWrapper, attention_kv_cache
from nano_vllm_x_amd.qwen3 import Qwen3Config, Qwen3ForCausalLM


def _model(hidden=1024, heads=4, inter=512, dtype=torch.bfloat16):
    m = Qwen3ForCausalLM(Qwen3Config.from_dict(dict(architectures=["Qwen3ForCausalLM"], vocab_size=64, hidden_size=hidden, intermediate_size=inter, num_hidden_layers=2,
                                                    num_attention_heads=heads, num_key_value_heads=2, head_dim=128, max_position_embeddings=32, rms_norm_eps=1e-6,
                                                    rope_theta=1e6, tie_word_embeddings=True, torch_dtype="bfloat16"))).to(dtype)
    m.finalize()
    return m


def _plain(m, x=None, wrapper=None, mode=ForwardMode.DECODE) -> bool:
    wrapper = wrapper or PagedDecodeWrapper()
    if isinstance(wrapper, PagedDecodeWrapper):
        wrapper.qkv_fused = getattr(wrapper, "asked", True)
    x = torch.zeros(4, m.config.hidden_size, dtype=m.lm_head.weight.dtype) if x is None else x
    with torch.inference_mode(), attention_kv_cache(m, AttentionMetadata(mode, None, None, wrapper)):
        return bool(m.model._plain_decode(x))


def test_a_stack_as_built_is_plain():
    m = _model()
    assert _plain(m) and _plain(m, torch.zeros(256, 1024).bfloat16()) and not _plain(m, torch.zeros(257, 1024).bfloat16())


@pytest.mark.parametrize("change", [plain_calls._own_forward, plain_calls._parametrise, plain_calls._tensor_class, plain_calls._scaling, plain_calls._eps, plain_calls._rope,
                                    plain_calls._activation, plain_calls._compiled, plain_calls._hook])
def test_a_changed_module_is_called(change):
    m = _model()
    change(m)
    assert not _plain(m)


def test_other_steps_formats_sizes_and_layouts_keep_the_modules():
    m = _model()
    x = torch.zeros(4, 1024).bfloat16()
    assert not _plain(m, x.float()) and not _plain(m, x[:, :256]) and not _plain(m, torch.zeros(1024, 4).bfloat16().t())
    assert not _plain(m, mode=ForwardMode.PREFILL) and not _plain(m, wrapper=PagedPrefillWrapper())
    w = PagedDecodeWrapper()
    w.run_qkv = lambda *a, **k: None
    assert not _plain(m, wrapper=w)
    w = PagedDecodeWrapper()
    w.asked = False                    # a plan without the new rows' slots: norm, rotation and scatter are a launch of their own
    assert not _plain(m, wrapper=w)
    assert not _plain(_model(dtype=torch.float16)) and not _plain(_model(hidden=512)) and not _plain(_model(heads=2)) and not _plain(_model(inter=768))
    for layer, name in ((0, "o_proj"), (1, "qkv_proj")):
        m = _model()
        p = getattr(m.model.layers[layer].self_attn, name)
        p.weight = nn.Parameter(torch.zeros(p.weight.shape[1], p.weight.shape[0]).bfloat16().t())
        assert not _plain(m), name


@pytest.mark.parametrize("kind", ["qkv", "o", "gate_up", "down"])
def test_rows_that_a_projection_leaves_to_the_library(kind, monkeypatch):
    m = _model()
    monkeypatch.setitem(qwen3.DECODE_LINEAR_MAX_ROWS, kind, 3)
    assert not _plain(m) and _plain(m, torch.zeros(3, 1024).bfloat16())


@pytest.mark.parametrize("args,what", [
    (dict(mode=3, out=True, residual=True, norm_weight=True), "no out"), (dict(mode=3, k_splits=2, residual=True, norm_weight=True), "no out"),
    (dict(mode=0, out=True, squares=True, eps=1e-6), "no out"), (dict(mode=1, k_splits=4, squares=True, eps=1e-6), "no out"),
    (dict(mode=0, residual=True), "residual and norm_weight"), (dict(mode=1, norm_weight=True), "residual and norm_weight"),
    (dict(mode=2, residual=True, norm_weight=True), "residual and norm_weight"), (dict(mode=0, squares=True, residual=True), "residual and norm_weight"),
    (dict(mode=3), "residual and norm_weight"), (dict(mode=3, residual=True), "residual and norm_weight"), (dict(mode=0, eps=1e-6), "eps")])
def test_an_argument_that_a_product_does_not_take_is_refused(args, what):
    t = torch.zeros(4, 1024).bfloat16()
    with pytest.raises(Exception, match=what):
        ops.linear_decode(t, torch.zeros(32, 1024).bfloat16(), **{k: t if v is True else v for k, v in args.items()})
