"""Decode steps whose layers are one launch (csrc/decode_chain.hip) against the oracle in float32, on the caches that the step finds."""
import pytest
import torch

from test_gpu_decode_chain import LAYERS, ROUNDINGS, _prefill, _runner, _sequences, _step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nan", [False, True])
@pytest.mark.parametrize("lengths", [(1,), (63,), (64,), (1030,), (40, 1), (1, 64, 700), (5, 6, 7, 8, 9), (1100, 1, 30, 128, 64, 65, 400, 2)])
def test_a_step_against_the_oracle(lengths, nan):
    """Whatever lies in slots of nobody's, NaN too, is not read: slot 0 among them, which stands in for tokens past a chunk's end."""
    from nano_vllm_x_amd import qwen3
    from oracle.attention_oracle import block_table_oracle
    from oracle.layers_oracle import rope_table_oracle
    from oracle.qwen3_oracle import logits_oracle, pack_weights_oracle, qwen3_forward_oracle

    r, seqs = _runner(8, 1200), _sequences(lengths, 6)
    for s in seqs:
        s.kv_indices = [1 + 2 * i for i in s.kv_indices]
    n_slots = 2 * (sum(lengths) + len(lengths)) + 1
    r.initialize_kv_cache(n_slots)
    _prefill(r, seqs)
    cache, used = r.kv_cache, torch.tensor([i for s in seqs for i in s.kv_indices[:-1]], device="cuda")
    if nan:
        free = torch.ones(n_slots, dtype=torch.bool, device="cuda")
        free[used] = False
        cache.k_cache[:, free], cache.v_cache[:, free] = torch.nan, torch.nan
    k, v = (c[:, :n_slots].float().cpu().nan_to_num() for c in (cache.k_cache, cache.v_cache))
    got = _step(r, seqs)
    assert r.stats["chain_steps"] == 1
    cfg = dict(num_attention_heads=16, num_key_value_heads=8, head_dim=128, rms_norm_eps=r.hf_config.rms_norm_eps)
    w = pack_weights_oracle({n: t.bfloat16().float() for n, t in qwen3.random_checkpoint(r.hf_config, 3)}, LAYERS)
    table = block_table_oracle([(len(s.token_ids), s.kv_indices, s.cached_kv_len) for s in seqs])
    rope = rope_table_oracle(128, r.hf_config.max_position_embeddings, r.hf_config.rope_theta)
    hidden = qwen3_forward_oracle(w, cfg, [s.token_ids[-1] for s in seqs], [len(s.token_ids) - 1 for s in seqs], k, v, table, rope)
    want = logits_oracle(w, hidden)
    # a rounding to bfloat16 is off by 2^-8 / sqrt(3) of the value at most in the mean; those of the layers, of the final norm and of the logits, independent of each other
    bound = 2.0 ** -8 / 3 ** 0.5 * (ROUNDINGS * LAYERS + 2) ** 0.5
    assert float((got.cpu() - want).norm() / want.norm()) < bound
    new = torch.tensor([s.kv_indices[-1] for s in seqs])
    for mine, theirs in ((cache.k_cache, k), (cache.v_cache, v)):
        mine, theirs = mine[:, new.cuda()].float().cpu(), theirs[:, new]
        assert float((mine - theirs).norm() / theirs.norm()) < bound
