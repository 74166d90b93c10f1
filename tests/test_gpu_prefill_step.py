"""Prefill steps of a Qwen3 model as the runner queues them (in one native call up to some 1500 tokens of this width, without module calls above) against the module
graph, which a hook on any of its modules brings back."""
import pytest
import torch

pytestmark = pytest.mark.gpu

LAYERS, ROUNDINGS = 2, 9      # 16-bit stores of a layer that another order of summation can turn: norms 2, qkv, q and k, read-out, o, activation, down


def _runner(dtype):
    from nano_vllm_x_amd.core.model_runner import ModelRunner
    from nano_vllm_x_amd.qwen3 import Qwen3Config

    cfg = Qwen3Config.from_dict(dict(architectures=["Qwen3ForCausalLM"], vocab_size=1024, hidden_size=1024, intermediate_size=3072, num_hidden_layers=LAYERS,
                                     num_attention_heads=16, num_key_value_heads=8, head_dim=128, max_position_embeddings=2048, rms_norm_eps=1e-6,
                                     rope_theta=1e6, tie_word_embeddings=True, torch_dtype=dtype))
    r = ModelRunner(model="random", max_bs=8, enforce_eager=True, context_len=2048, config=cfg, dtype=dtype)
    r.load_model()
    r.initialize_kv_cache(4096)
    return r


def _step(r, lens, cached):
    """Logits of the last tokens and the cache rows of the last layer after one step of prompts of `lens` new tokens behind `cached` ones."""
    from nano_vllm_x_amd.core.common import ForwardBatch, ForwardMode, Sequence

    gen = torch.Generator().manual_seed(sum(lens) + cached)
    r.kv_cache.k_cache.copy_(torch.randn(r.kv_cache.k_cache.shape, generator=gen).to(r.dtype) * 0.1)
    r.kv_cache.v_cache.copy_(torch.randn(r.kv_cache.v_cache.shape, generator=gen).to(r.dtype) * 0.1)
    slots = torch.randperm(4096, generator=gen).tolist()
    seqs, at = [], 0
    for i, n in enumerate(lens):
        ids = torch.randint(0, 1024, (n + cached,), generator=gen).tolist()
        seqs.append(Sequence(seq_id=str(i), token_ids=ids, num_tokens=len(ids), prompt_len=len(ids), kv_indices=slots[at:at + len(ids)], cached_kv_len=cached))
        at += len(ids)
    logits = r.compute_logits(ForwardBatch(forward_mode=ForwardMode.PREFILL, num_seqs=len(seqs), seqs=seqs))
    return logits.float(), r.kv_cache.k_cache[-1].float(), r.kv_cache.v_cache[-1].float()


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("lens,cached", [((1,), 0), ((1, 1, 1), 7), ((255,), 0), ((256,), 3), ((257,), 0), ((300, 5, 206), 64), ((600,), 0), ((1100,), 0), ((1530,), 0), ((1500, 20, 100), 100)])
def test_prefill_steps_equal_the_module_graph(dtype, lens, cached):
    r = _runner(dtype)
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
def test_a_prompt_s_logits_do_not_depend_on_what_shares_its_step(alone):
    """Whatever tile a step's size chooses, a row's sums run in the same order: the same bits alone and among 256, 500, 1000 and 3000 other tokens."""
    r = _runner("bfloat16")
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
