"""Products of decode steps that carry the residual sum and norm between two of them (ops.linear_decode with mode 3 and with squares), against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _case(rows, hidden, k, n, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g)
    return r(rows, k).to(BF), (r(hidden, k) * k ** -0.5).to(BF), (3 * r(rows, hidden)).to(BF), (1 + 0.2 * r(hidden)).to(BF), (r(n, hidden) * hidden ** -0.5).to(BF)


@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17, 32, 33, 48, 49, 111, 112, 128, 129, 200, 256])
@pytest.mark.parametrize("hidden,k,n", [(1024, 512, 32), (1024, 2048, 4096), (1024, 3072, 6144), (1024, 2560, 1056)])
def test_norm_between_two_products(rows, hidden, k, n):
    from nano_vllm_x_amd import ops

    x, w, res, nw, w2 = _case(rows, hidden, k, n, rows + k)
    c = [t.cuda() for t in (x, w, res, nw, w2)]
    with torch.inference_mode():
        h, new, squares = ops.linear_decode(c[0], c[1], mode=3, residual=c[2], norm_weight=c[3])
        plain = ops.linear_decode(h, c[4], mode=0, squares=squares, eps=1e-6)
        act = ops.linear_decode(h, c[4], mode=1, squares=squares, eps=1e-6)
    # the product rounds to bfloat16 (2^-9 of it) before the residual is added, as a product of its own; the new residual rounds once more
    prod = x.double() @ w.double().T
    s = prod.to(BF).double() + res.double()
    slack = 2.0 ** -8 * prod.abs() + k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((new.cpu().double() - s).abs() <= slack + 2.0 ** -8 * s.abs()).all())
    assert bool(((h.cpu().double() - s * nw.double()).abs() <= (slack + 2.0 ** -8 * s.abs()) * nw.double().abs()).all())
    assert squares.shape[0] == -(-rows // 32) * 32 and hidden % squares.shape[1] == 0
    by_tile = lambda t: t.view(rows, squares.shape[1], -1).sum(2)
    assert bool(((squares[:rows].cpu().double() - by_tile(s * s)).abs() <= by_tile(2 * slack * s.abs() + slack ** 2 + 64 * 2.0 ** -24 * s * s)).all())
    # of the rows that the first product gave: h and the squares carry one rounding each
    hd, inv = h.cpu().double(), 1 / torch.sqrt(squares[:rows].cpu().double().sum(1, keepdim=True) / hidden + 1e-6)
    y = (hd @ w2.double().T) * inv
    near = hidden * 2.0 ** -23 * (hd.abs() @ w2.double().abs().T) * inv
    assert bool(((plain.cpu().double() - y).abs() <= 2.0 ** -8 * y.abs() + near).all())
    gate, up = y.to(BF).double().chunk(2, 1)
    want = torch.nn.functional.silu(gate) * up
    # each of gate and up may round the other way (2^-8), silu rounds (2^-8) and so does the product; |silu'| <= 1.1
    gs, us = (2.0 ** -8 * y.abs() + near).chunk(2, 1)
    bound = (1.1 * gs + 2.0 ** -8 * torch.nn.functional.silu(gate).abs()) * (up.abs() + us) + torch.nn.functional.silu(gate).abs() * us + 2.0 ** -8 * want.abs() + 1e-30
    assert bool(((act.cpu().double() - want).abs() <= bound).all())


@pytest.mark.parametrize("k", [2048, 3072])
def test_a_row_s_result_does_not_depend_on_the_number_of_rows(k):
    """(A batch may be replayed from a larger batch's graph.)"""
    from nano_vllm_x_amd import ops

    x, w, res, nw, w2 = (t.cuda() for t in _case(256, 1024, k, 2048, 9))
    first = None
    with torch.inference_mode():
        for rows in (1, 8, 9, 16, 17, 32, 33, 48, 49, 64, 65, 111, 112, 128, 129, 255, 256):
            h, new, squares = ops.linear_decode(x[:rows], w, mode=3, residual=res[:rows], norm_weight=nw)
            got = (h[0], new[0], ops.linear_decode(h, w2, mode=0, squares=squares, eps=1e-6)[0], ops.linear_decode(h, w2, mode=1, squares=squares, eps=1e-6)[0])
            first = first or got
            assert all(torch.equal(a, b) for a, b in zip(first, got)), rows


def test_operands_that_the_kernels_do_not_read_are_refused():
    from nano_vllm_x_amd import ops

    x, w, res, nw, w2 = (t.cuda() for t in _case(4, 1024, 2048, 512, 3))
    for args in (dict(residual=res.half(), norm_weight=nw), dict(residual=res, norm_weight=nw[:512]), dict(residual=res.t().contiguous().t(), norm_weight=nw)):
        with pytest.raises(Exception):
            ops.linear_decode(x, w, mode=3, **args)
    h, _, squares = ops.linear_decode(x, w, mode=3, residual=res, norm_weight=nw)
    for bad in (squares[:4], squares.double()):
        with pytest.raises(Exception):
            ops.linear_decode(h, w2, mode=0, squares=bad, eps=1e-6)
    for m in (1, 16, 257):
        assert ops.decode_boundary_fits(m, 1024, 2048, 3072, BF) == (m <= ops.BOUNDARY_ROWS)
    assert not ops.decode_boundary_fits(4, 512, 2048, 3072, BF) and not ops.decode_boundary_fits(4, 1024, 2048, 3072, torch.float16)


LAYERS, ROUNDINGS = 2, 9      # 16-bit stores of a layer that another order of summation can turn: norms 2, qkv, q and k, read-out, o, activation, down


@pytest.mark.parametrize("rows", [3, 20, 40, 100, 150, 256])
def test_a_model_s_decode_step_with_and_without(rows, monkeypatch):
    """The step queued past its modules against the module graph (which a hook asks for), caches included: as many roundings, some in other places."""
    from nano_vllm_x_amd import ops, qwen3
    from nano_vllm_x_amd.core.common import ForwardBatch, ForwardMode, Sequence
    from nano_vllm_x_amd.core.model_runner import ModelRunner

    cfg = qwen3.Qwen3Config(vocab_size=512, hidden_size=1024, intermediate_size=1536, num_hidden_layers=LAYERS, num_attention_heads=4, num_key_value_heads=2, head_dim=128,
                            max_position_embeddings=256)
    out, hooks, modes, product = [], [], [], ops.linear_decode
    monkeypatch.setattr(ops, "linear_decode", lambda *a, mode=0, **k: (modes.append((mode, "squares" in k)), product(*a, mode=mode, **k))[1])
    for hooked in (False, True):
        r = ModelRunner(model="mid", max_bs=256, enforce_eager=True, context_len=64, config=cfg, seed=3)
        r.load_model()
        r.initialize_kv_cache(rows * 8)
        seqs = [Sequence(seq_id=f"m{i}", token_ids=[(7 * i + j) % 512 for j in range(4)], num_tokens=4, prompt_len=4, kv_indices=list(range(8 * i, 8 * i + 4))) for i in range(rows)]
        r.compute_logits(ForwardBatch(forward_mode=ForwardMode.PREFILL, num_seqs=rows, seqs=seqs))
        for i, s in enumerate(seqs):
            s.cached_kv_len, s.token_ids, s.kv_indices = 4, s.token_ids + [i], s.kv_indices + [8 * i + 4]
        if hooked:
            r.model.model.layers[1].mlp.register_forward_hook(lambda *a: hooks.append(1))
        modes.clear()
        logits = r.compute_logits(ForwardBatch(forward_mode=ForwardMode.DECODE, num_seqs=rows, seqs=seqs))
        # every norm but the first and the last rides on the products around it, or none does
        assert [modes.count((3, False)), modes.count((1, True)), modes.count((0, True))] == ([0, 0, 0] if hooked else [2 * LAYERS - 1, LAYERS, LAYERS - 1])
        out.append((logits.float(), r.kv_cache.k_cache[-1].float(), r.kv_cache.v_cache[-1].float()))
    assert len(hooks) == 1
    # every rounding that turns is a unit of the last place, uniform within it: 2^-8 / sqrt(3) of the value at most, both sides' and all layers' independent of
    # each other, the LM head's on top
    bound = 2.0 ** -8 / 3 ** 0.5 * (2 * (ROUNDINGS * LAYERS + 1)) ** 0.5
    for a, b in zip(*out):
        assert bool(torch.isfinite(a).all()) and float((a - b).norm() / b.norm()) < bound
