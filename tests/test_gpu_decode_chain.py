"""Decode steps whose layers are one launch (csrc/decode_chain.hip) against the same steps launch by launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu
LAYERS, ROUNDINGS = 3, 9      # 16-bit stores of a layer that another order of summation can turn: norms 2, qkv, q and k, read-out, o, activation, down


def _runner(max_bs, context, layers=LAYERS):
    from nano_vllm_x_amd import qwen3
    from nano_vllm_x_amd.core.model_runner import ModelRunner

    cfg = qwen3.Qwen3Config(vocab_size=512, hidden_size=1024, intermediate_size=3072, num_hidden_layers=layers, num_attention_heads=16, num_key_value_heads=8, head_dim=128,
                            max_position_embeddings=2048)
    r = ModelRunner(model="mid", max_bs=max_bs, context_len=context, config=cfg, seed=3)
    r.load_model()
    return r


def _sequences(lengths, seed=0):
    """Prompts of these lengths in slots that lie in no order, and one token more."""
    from nano_vllm_x_amd.core.common import Sequence

    g = torch.Generator().manual_seed(seed)
    slots, seqs, at = torch.randperm(sum(lengths) + len(lengths), generator=g).tolist(), [], 0
    for i, n in enumerate(lengths):
        ids = torch.randint(512, (n + 1,), generator=g).tolist()
        seqs.append(Sequence(seq_id=f"c{seed}.{i}", token_ids=ids, num_tokens=n + 1, prompt_len=n, kv_indices=slots[at:at + n + 1]))
        at += n + 1
    return seqs


def _step(r, seqs):
    from nano_vllm_x_amd.core.common import ForwardBatch, ForwardMode

    return r.compute_logits(ForwardBatch(forward_mode=ForwardMode.DECODE, num_seqs=len(seqs), seqs=seqs)).float()


def _prefill(r, seqs):
    from nano_vllm_x_amd.core.common import ForwardBatch, ForwardMode

    full = [(s.token_ids, s.kv_indices) for s in seqs]
    for s in seqs:
        s.token_ids, s.kv_indices, s.cached_kv_len = s.token_ids[:-1], s.kv_indices[:-1], 0
    r.compute_logits(ForwardBatch(forward_mode=ForwardMode.PREFILL, num_seqs=len(seqs), seqs=seqs))
    for s, (ids, slots) in zip(seqs, full):
        s.token_ids, s.kv_indices, s.cached_kv_len = ids, slots, len(ids) - 1


@pytest.mark.parametrize("lengths", [(1,), (62,), (63,), (64,), (65,), (127,), (1030,), (40, 1), (1023, 200), (1, 64, 700), (300, 2, 129, 64), (5, 6, 7, 8, 9), (200, 1, 1, 90, 500, 63),
                                     (64,) * 7, (1100, 1, 30, 128, 64, 65, 400, 2)])
def test_one_launch_against_many(lengths):
    r = _runner(len(lengths), 1200)
    r.initialize_kv_cache(sum(lengths) + len(lengths))
    assert r.decode_chain is not None
    seqs, cache, out = _sequences(lengths), r.kv_cache, []
    _prefill(r, seqs)
    new = torch.tensor([s.kv_indices[-1] for s in seqs], device="cuda")
    for chain in (None, r.chain_graph):
        r.chain_graph = chain
        cache.k_cache[:, new], cache.v_cache[:, new] = 0, 0
        logits = _step(r, seqs)
        out.append((logits, cache.k_cache.float(), cache.v_cache.float()))
    assert r.stats["chain_steps"] == 1 and not r.decode_chain._status[0]
    # every rounding that turns is a unit of the last place, uniform within it: 2^-8 / sqrt(3) of the value at most, both sides' and all layers' independent of
    # each other, the LM head's on top
    bound = 2.0 ** -8 / 3 ** 0.5 * (2 * (ROUNDINGS * LAYERS + 1)) ** 0.5
    for a, b in zip(*out):
        assert bool(torch.isfinite(a).all()) and bool(torch.isfinite(b).all()) and float((a - b).norm() / b.norm()) < bound
    for a, b in zip(out[0][1:], out[1][1:]):      # only the new rows were written, and those of the first layer hang on nothing that differs
        keep = torch.ones(a.shape[1], dtype=torch.bool, device="cuda")
        keep[new] = False
        assert torch.equal(a[:, keep], b[:, keep]) and torch.equal(a[0], b[0]) and bool((a[:, new].abs().sum((2, 3)) > 0).all())


def test_replays_among_other_work():
    """Batches of several sizes in turn, each several times with eager work between: every replay gives what the first gave, and that, padded rows beside it or not (three
    go as four, five as eight), is what the layers launch by launch give."""
    r = _runner(8, 300)
    lengths = (100, 7, 250, 64, 31, 128, 1, 199)
    r.initialize_kv_cache(sum(lengths) + len(lengths))
    seqs = _sequences(lengths, 1)
    _prefill(r, seqs)
    first = {}
    for turn in range(3):
        for n in (1, 3, 8, 2, 5, 4):
            got = _step(r, seqs[:n])
            torch.randn(1 << 20, device="cuda").sum().item()
            first.setdefault(n, got)
            assert torch.equal(first[n], got), (turn, n)
    assert r.stats["chain_steps"] == 18 and r.stats["graph_steps"] == 18
    r.decode_chain.check()
    r.chain_graph = None
    bound = 2.0 ** -8 / 3 ** 0.5 * (2 * (ROUNDINGS * LAYERS + 1)) ** 0.5      # (as above)
    for n, got in first.items():
        want = _step(r, seqs[:n])
        assert got.shape == want.shape and float((got - want).norm() / want.norm()) < bound, n


def test_more_tokens_than_pay_take_the_launches():
    from nano_vllm_x_amd import ops

    assert ops.DecodeChain.faster(8, 10000) and not ops.DecodeChain.faster(8, 10001) and not ops.DecodeChain.faster(9, 10)
    r = _runner(5, 2000)
    r.initialize_kv_cache(5 * 1800)
    seqs = _sequences((1750,) * 5, 2)
    _prefill(r, seqs[:5])
    r.decode_chain.faster = lambda rows, tokens: ops.DecodeChain.faster(rows, tokens + 2000)
    _step(r, seqs)
    assert "chain_steps" not in r.stats and r.stats["graph_steps"] == 1


def test_three_on_a_device_take_turns():
    """(There is room for two at once.)"""
    runners, want = [_runner(2, 200) for _ in range(3)], None
    streams, seqs = [torch.cuda.Stream() for _ in runners], _sequences((100, 150), 3)
    for r in runners:
        r.initialize_kv_cache(252)
        for s in seqs:
            s.cached_kv_len = 0
        _prefill(r, seqs)
    torch.cuda.synchronize()
    got = []
    for _ in range(4):
        for r, st in zip(runners, streams):
            with torch.cuda.stream(st):
                got.append(_step(r, seqs))
    torch.cuda.synchronize()
    for r in runners:
        r.decode_chain.check()
        assert r.stats["chain_steps"] == 4
    assert all(torch.equal(got[0], g) for g in got)


def test_the_words_are_cleared_before_their_marks_come_round():
    """Marks of 32 bits: the count starts anew long before, with words that carry none."""
    from nano_vllm_x_amd import ops

    assert ops.DecodeChain.STEPS * ops.DecodeChain.LAYERS <= 1 << 31
    r = _runner(4, 300)
    lengths = (100, 7, 250, 64)
    r.initialize_kv_cache(sum(lengths) + len(lengths))
    seqs, chain = _sequences(lengths, 1), r.decode_chain
    _prefill(r, seqs)
    want = {n: _step(r, seqs[:n]) for n in (1, 4)}
    torch.cuda.synchronize()
    # as after so many steps of one sequence: the other rows' words still carry what they were left with, here the marks of the steps to come
    chain.steps = chain.STEPS - 1
    chain.words.copy_((1 + torch.arange(chain.words.numel(), device="cuda") % (2 * LAYERS)) << 32)
    chain.epoch[:1].fill_(1 << 20)
    for n, epoch in ((1, (1 << 20) + LAYERS), (4, 1 + LAYERS), (1, 1 + 2 * LAYERS)):
        assert torch.equal(_step(r, seqs[:n]), want[n])
        torch.cuda.synchronize()
        assert chain.epoch.tolist() == [epoch, 0]
    assert chain.steps == 2
