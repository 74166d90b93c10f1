"""Prefill steps of a Qwen3 model as the runner queues them (in one native call up to 4096 tokens of this width, without module calls above) against the module
graph, which a hook on any of its modules brings back."""
import pytest
import torch

pytestmark = pytest.mark.gpu

LAYERS, ROUNDINGS = 2, 9      # 16-bit stores of a layer that another order of summation can turn: norms 2, qkv, q and k, read-out, o, activation, down


def _runner(dtype, hidden=1024, inter=3072, heads=16, slots=4096):
    from nano_vllm_x_amd.core.model_runner import ModelRunner
    from nano_vllm_x_amd.qwen3 import Qwen3Config

    cfg = Qwen3Config.from_dict(dict(architectures=["Qwen3ForCausalLM"], vocab_size=1024, hidden_size=hidden, intermediate_size=inter, num_hidden_layers=LAYERS,
                                     num_attention_heads=heads, num_key_value_heads=8, head_dim=128, max_position_embeddings=2048, rms_norm_eps=1e-6,
                                     rope_theta=1e6, tie_word_embeddings=True, torch_dtype=dtype))
    r = ModelRunner(model="random", max_bs=8, enforce_eager=True, context_len=2048, config=cfg, dtype=dtype)
    r.load_model()
    r.initialize_kv_cache(slots)
    return r


@pytest.fixture
def route(monkeypatch):
    """How often a step went out natively, and how often a long step took SiluAndMul into its product."""
    from nano_vllm_x_amd import ops

    calls = {"native": 0, "gated": 0}

    def counted(name, fn):
        def run(*args):
            out = fn(*args)
            calls[name] += out is not None
            return out
        return run

    monkeypatch.setattr(ops, "prefill_step", counted("native", ops.prefill_step))
    monkeypatch.setattr(ops, "gated_product", counted("gated", ops.gated_product))
    return calls


def _step(r, lens, cached):
    """Logits of the last tokens and the cache rows of the last layer after one step of prompts of `lens` new tokens behind `cached` ones."""
    from nano_vllm_x_amd.core.common import ForwardBatch, ForwardMode, Sequence

    gen = torch.Generator().manual_seed(sum(lens) + cached)
    r.kv_cache.k_cache.copy_(torch.randn(r.kv_cache.k_cache.shape, generator=gen).to(r.dtype) * 0.1)
    r.kv_cache.v_cache.copy_(torch.randn(r.kv_cache.v_cache.shape, generator=gen).to(r.dtype) * 0.1)
    slots = torch.randperm(r.kv_cache.k_cache.shape[1], generator=gen).tolist()
    seqs, at = [], 0
    for i, n in enumerate(lens):
        ids = torch.randint(0, 1024, (n + cached,), generator=gen).tolist()
        seqs.append(Sequence(seq_id=str(i), token_ids=ids, num_tokens=len(ids), prompt_len=len(ids), kv_indices=slots[at:at + len(ids)], cached_kv_len=cached))
        at += len(ids)
    logits = r.compute_logits(ForwardBatch(forward_mode=ForwardMode.PREFILL, num_seqs=len(seqs), seqs=seqs))
    return logits.float(), r.kv_cache.k_cache[-1].float(), r.kv_cache.v_cache[-1].float()


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("lens,cached", [((1,), 0), ((1, 1, 1), 7), ((255,), 0), ((256,), 3), ((257,), 0), ((300, 5, 206), 64), ((600,), 0), ((1100,), 0), ((1530,), 0), ((1500, 20, 100), 100)])
def test_prefill_steps_equal_the_module_graph(dtype, lens, cached, route):
    _equal_to_the_module_graph(_runner(dtype), dtype, lens, cached)
    assert route == {"native": 1, "gated": 0}


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("lens,cached,limit", [((2000, 2000, 97), 0, None), ((2000, 1, 2000, 500), 40, None), ((1, 1, 1), 7, 0), ((300, 5, 206), 64, 0), ((1100,), 0, 0)])
def test_long_steps_equal_the_module_graph(dtype, lens, cached, limit, route, monkeypatch):
    """Steps past the native call's limit, and shorter ones with the limit taken down."""
    from nano_vllm_x_amd import qwen3

    if limit is not None:
        monkeypatch.setattr(qwen3, "PREFILL_STEP_MAX_WORK", limit)
        monkeypatch.setattr(qwen3, "PREFILL_STEP_MAX_WORK_NARROW", limit)
    _equal_to_the_module_graph(_runner(dtype, slots=8192), dtype, lens, cached)
    assert route == {"native": 0, "gated": LAYERS}


def _equal_to_the_module_graph(r, dtype, lens, cached):
    got = _step(r, lens, cached)
    hook = r.model.model.layers[1].mlp.register_forward_hook(lambda *_: None)
    ref = _step(r, lens, cached)
    hook.remove()
    # every rounding that turns is one unit of the last place, uniform within it: 2^-8 (2^-11) / sqrt(3) of the value at most, both sides' and
    # all layers' independent of each other; a norm behind a sum hands on what the rows hold, the LM head adds its rounding
    ulp = 2.0 ** (-8 if dtype == "bfloat16" else -11)
    bound = ulp / 3 ** 0.5 * (2 * (ROUNDINGS * LAYERS + 1)) ** 0.5
    for a, b in zip(got, ref):
        assert torch.isfinite(a).all()
        assert float((a - b).norm() / b.norm()) < bound


@pytest.mark.parametrize("alone", [1, 33, 65, 200])
def test_a_prompt_s_logits_do_not_depend_on_what_shares_its_step(alone, route, monkeypatch):
    """Whatever tile a step's size chooses, a row's sums run in the same order: the same bits alone and among 256, 500, 1000 and 3000 other tokens, and among 4500
    and, with the native call's limit taken down, 600 and 2000 (through the library's products, which take K in that order too for steps of such sizes)."""
    from nano_vllm_x_amd import qwen3

    r = _runner("bfloat16", slots=8192)
    gen = torch.Generator().manual_seed(alone)
    ids = torch.randint(0, 1024, (alone,), generator=gen).tolist()

    def first(others):
        from nano_vllm_x_amd.core.common import ForwardBatch, ForwardMode, Sequence

        prompts = [ids] + [torch.randint(0, 1024, (n,), generator=gen).tolist() for n in others]
        at, seqs = 0, []
        for i, p in enumerate(prompts):
            seqs.append(Sequence(seq_id=str(i), token_ids=p, num_tokens=len(p), prompt_len=len(p), kv_indices=list(range(at, at + len(p)))))
            at += len(p)
        return r.compute_logits(ForwardBatch(forward_mode=ForwardMode.PREFILL, num_seqs=len(seqs), seqs=seqs))[0]

    want = first([])
    for others in ([256], [500], [400, 600], [1500, 1500]):
        assert torch.equal(first(others), want), others
    assert route == {"native": 5, "gated": 0}
    assert torch.equal(first([2000, 2000, 500]), want)
    monkeypatch.setattr(qwen3, "PREFILL_STEP_MAX_WORK", 0)
    monkeypatch.setattr(qwen3, "PREFILL_STEP_MAX_WORK_NARROW", 0)
    for others in ([600], [2000]):
        assert torch.equal(first(others), want), others
    assert route == {"native": 5, "gated": 3 * LAYERS}


@pytest.mark.parametrize("alone", [1, 33, 100])
def test_a_prompt_s_rows_at_the_sizes_of_8b_do_not_depend_on_what_shares_a_native_step(alone):
    """Layers of 4096: steps of up to 124 tokens are the native call's, whose sums run in one order whatever the tile (longer ones are the library's,
    which promises nothing of the sort).  The cache rows of the last layer hold all products of the layers before it."""
    from nano_vllm_x_amd.core.common import ForwardBatch, ForwardMode, Sequence

    r = _runner("bfloat16", hidden=4096, inter=12288, heads=32)
    gen = torch.Generator().manual_seed(alone)
    ids = torch.randint(0, 1024, (alone,), generator=gen).tolist()

    def rows(others):
        prompts = [ids] + [torch.randint(0, 1024, (n,), generator=gen).tolist() for n in others]
        at, seqs = 0, []
        for i, p in enumerate(prompts):
            seqs.append(Sequence(seq_id=str(i), token_ids=p, num_tokens=len(p), prompt_len=len(p), kv_indices=list(range(at, at + len(p)))))
            at += len(p)
        r.compute_logits(ForwardBatch(forward_mode=ForwardMode.PREFILL, num_seqs=len(seqs), seqs=seqs))
        return r.kv_cache.k_cache[-1][:alone].clone(), r.kv_cache.v_cache[-1][:alone].clone()

    want = rows([])
    assert all(bool(x.float().abs().sum() > 0) for x in want)
    for others in ([1], [7, 9], [24], [124 - alone]):
        for got, expected in zip(rows(others), want):
            assert torch.equal(got, expected), others


class _Doubled(torch.nn.Linear):
    def forward(self, x):
        return 2 * super().forward(x)


def _replaced(layer):
    lin, w = _Doubled(3072, 1024, bias=False), layer.mlp.down_proj.weight
    lin.weight = w
    layer.mlp.down_proj = lin


def _with_bias(layer):
    layer.self_attn.qkv_proj.bias = torch.nn.Parameter(torch.ones(4096, device="cuda", dtype=layer.mlp.down_proj.weight.dtype))


def _parametrised(layer):
    class Half(torch.nn.Module):
        def forward(self, w):
            return 0.5 * w

    torch.nn.utils.parametrize.register_parametrization(layer.self_attn.o_proj, "weight", Half())


def _other_scaling(layer):
    layer.self_attn.attn.scaling = 0.02


def _off_border(layer):
    w = layer.mlp.gate_up_proj.weight
    flat = torch.empty(w.numel() + 1, dtype=w.dtype, device="cuda")
    flat[1:] = w.detach().reshape(-1)
    layer.mlp.gate_up_proj.weight = torch.nn.Parameter(flat[1:].view_as(w))


def _pruned(layer):
    g, d = layer.mlp.gate_up_proj, layer.mlp.down_proj
    g.weight = torch.nn.Parameter(torch.cat([g.weight[:2048], g.weight[3072:5120]]))
    d.weight = torch.nn.Parameter(d.weight[:, :2048].contiguous())


@pytest.mark.parametrize("change", [_replaced, _with_bias, _parametrised, _other_scaling, _off_border, _pruned])
def test_what_a_user_changed_in_a_layer_counts(change):
    """Modules replaced, parametrised, given a bias or a scale, weights off a 16-byte border or of a pruned layer: the bits of the module graph."""
    r = _runner("bfloat16")
    plain = _step(r, (300, 5), 10)[0]
    with torch.no_grad():
        change(r.model.model.layers[1])
    got = _step(r, (300, 5), 10)
    hook = r.model.model.layers[1].mlp.register_forward_hook(lambda *_: None)
    ref = _step(r, (300, 5), 10)
    hook.remove()
    assert all(torch.equal(a, b) for a, b in zip(got, ref))
    assert change is _off_border or not torch.equal(got[0], plain)
