"""The sampler's paths against each other: rows kept on the compute unit (16-byte aligned bfloat16 rows) and the general kernel draw the same tokens
for the same logits, whatever survives the filters: nothing but the maximum, a few tokens, as many as the list of survivors holds, more."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _draw(lg, T, k, p, m, seed):
    from nano_vllm_x_amd import ops

    return ops.sample(lg, T, k, p, m, seed, 5).cpu()


@pytest.mark.parametrize("vocab", [8, 4096, 8192 * 3 + 8, 151936, 155648])
@pytest.mark.parametrize("rows", [1, 33, 130, 300])
def test_aligned_and_unaligned_rows_draw_the_same(vocab, rows):
    if rows > 33 and vocab > 100000:
        rows = 40
    g = torch.Generator(device="cuda").manual_seed(vocab + rows)
    lg = (2.5 * torch.randn((rows, vocab), generator=g, device="cuda")).to(torch.bfloat16)
    if rows > 8:
        lg[3], lg[4, vocab // 2:], lg[5] = 0.0, float("-inf"), lg[5].round()
    wide = torch.empty((rows, vocab + 1), dtype=torch.bfloat16, device="cuda")      # odd row stride: the general kernel, token by token
    wide[:, :vocab] = lg
    r = torch.arange(rows, device="cuda")
    T = 0.4 + 0.2 * (r % 5).float()
    T[r % 13 == 12] = 0.0
    off = lambda x: torch.full((rows,), x, device="cuda")
    every, one, none = off(vocab).long(), off(1.0), off(0.0)
    for k, p, m in ((every, one, none), (every, one, off(1.0)), (every, one, off(0.999)), (every, one, off(0.05)), (every, one, off(1e-9)), (every, one, off(1.5)),
                    (every, off(1e-6), none), (every, off(0.5), none), (every, off(0.9), none), (every, off(0.9999), none), (off(1).long(), one, none),
                    (off(50).long(), off(0.9), off(0.05)), (torch.where(r % 2 == 0, 20, vocab), torch.where(r % 3 == 0, 0.8, 1.0), torch.where(r % 5 == 0, 0.1, 0.0))):
        assert torch.equal(_draw(lg, T, k, p, m, 3), _draw(wide[:, :vocab], T, k, p, m, 3))


@pytest.mark.parametrize("shape", ["negative", "nearly equal", "wide", "all equal", "few values", "infinite"])
def test_boundaries_outside_the_largest_scores_draw_the_same(shape):
    """Boundaries among the 2048 largest scores and below them, masses of neither kind, more than a thousand ties at the boundary, survivors that fill the list:
    the general kernel's tokens."""
    rows, vocab = 24, 65536
    g = torch.Generator(device="cuda").manual_seed(len(shape))
    x = torch.randn((rows, vocab), generator=g, device="cuda")
    lg = {"negative": -x.abs() - 1e-4, "nearly equal": 1e-5 * x, "wide": torch.sign(x) * torch.exp(6 * x - 12), "all equal": 0 * x + 1.5, "few values": x.round(),
          "infinite": torch.where(x > 4, float("inf"), torch.where(x < -2, float("-inf"), x))}[shape].to(torch.bfloat16)
    wide = torch.empty((rows, vocab + 1), dtype=torch.bfloat16, device="cuda")
    wide[:, :vocab] = lg
    T = 0.05 + 0.25 * (torch.arange(rows, device="cuda") % 6).float()
    off = lambda v, d=torch.float32: torch.full((rows,), v, dtype=d, device="cuda")
    for k in (vocab, 3, 1000, 30000, vocab - 1):
        for p in (1.0, 0.999, 0.9, 0.4, 1e-4):
            for m in (0.0, 0.3):
                a = (off(k, torch.int64), off(p), off(m))
                assert torch.equal(_draw(lg, T, *a, 3), _draw(wide[:, :vocab], T, *a, 3)), (k, p, m)


@pytest.mark.parametrize("shape", ["below zero", "one above", "few above", "around zero", "grid", "small", "large"])
def test_boundaries_among_negative_scores_draw_the_same(shape):
    """Largest scores above zero, boundaries below it, above and below the negative scores that are counted, and in between: the general kernel's tokens."""
    rows, vocab = 24, 65536
    g = torch.Generator(device="cuda").manual_seed(7 * len(shape))
    x = torch.randn((rows, vocab), generator=g, device="cuda")
    few = torch.rand((rows, vocab), generator=g, device="cuda") < 2e-4
    lg = {"below zero": 2.5 * x - 8, "one above": torch.where(x == x.max(1, keepdim=True).values, 0.75, 0.5 * x - 30), "few above": torch.where(few, x.abs(), x - 12),
          "around zero": torch.where(few, 3.0, 1e-4 * x), "grid": (4 * x).round() / 2 - 6, "small": torch.where(few, 0.01, -x.abs() / 100),
          "large": torch.where(few, 1e4, -1e4 * x.abs())}[shape].to(torch.bfloat16)
    assert bool((lg.float().max(1).values > 0).all())
    wide = torch.empty((rows, vocab + 1), dtype=torch.bfloat16, device="cuda")
    wide[:, :vocab] = lg
    T = torch.tensor([0.05, 0.3, 0.8, 1.0, 2.0, 40.0], device="cuda").repeat(rows // 6)
    off = lambda v, d=torch.float32: torch.full((rows,), v, dtype=d, device="cuda")
    for k in (vocab, 1, 20, 200, 30000, vocab - 1):
        for p in (1.0, 0.999, 0.9, 0.4):
            for m in (0.0, 0.05):
                a = (off(k, torch.int64), off(p), off(m))
                assert torch.equal(_draw(lg, T, *a, 3), _draw(wide[:, :vocab], T, *a, 3)), (k, p, m)


@pytest.mark.parametrize("vocab", [32000, 151936])
@pytest.mark.parametrize("score", [4.0, -4.0])
def test_ties_at_the_boundary_are_parted_alike(vocab, score):
    """One to thousands of tokens with the boundary's score, from none to all of them dropped: the general kernel's tokens, by a list of up to 384 or by passes."""
    counts = (1, 2, 63, 382, 384, 385, 1024, 1025, 9000)
    g = torch.Generator().manual_seed(vocab)
    lg, tops = torch.full((3 * len(counts), vocab), -40.0), []
    for i, n in enumerate(counts):
        for j, share in enumerate((0.02, 0.5, 0.999)):       # of the ties' mass that is kept
            at = torch.randperm(vocab, generator=g)[:n + 3]
            lg[3 * i + j, at[:3]], lg[3 * i + j, at[3:]] = 4.5, score
            above, ties = 3 * 2.718281828 ** (4.5 - score), n
            tops.append((above + share * ties) / (above + ties))
    lg = lg.to(torch.bfloat16).cuda()
    wide = torch.empty((lg.shape[0], vocab + 1), dtype=torch.bfloat16, device="cuda")
    wide[:, :vocab] = lg
    p, one = torch.tensor(tops, device="cuda"), torch.ones(lg.shape[0], device="cuda")
    for k in (vocab, vocab - 1):
        for step in range(8):
            a = (torch.full((lg.shape[0],), k, device="cuda"), p, 0 * one)
            assert torch.equal(_draw(lg, one, *a, step), _draw(wide[:, :vocab], one, *a, step)), (k, step)


def test_min_p_keeps_the_tokens_of_its_ratio():
    """Among logits 0, -1, -2, ... at temperature 1 the ratio of a probability to the largest is e^-i: min_p between e^-3 and e^-2 leaves three tokens."""
    lg = torch.full((64, 1024), -100.0, device="cuda", dtype=torch.bfloat16)
    lg[:, 100:108] = -torch.arange(8, device="cuda").to(torch.bfloat16)
    z = lambda v, d=torch.float32: torch.full((64,), v, device="cuda", dtype=d)
    seen = set()
    for seed in range(60):
        seen |= set(_draw(lg, z(1.0), z(1024, torch.int64), z(1.0), z(0.09), seed).tolist())
    assert seen == {100, 101, 102}      # (the rarest of the three is drawn with probability 0.09: 3840 draws miss it with 1e-157)


@pytest.mark.parametrize("vocab", [9999, 24584, 50257, 100352])
@pytest.mark.parametrize("rows", [5, 17, 64, 96, 128, 200, 256])
def test_slices_do_not_change_the_draw(rows, vocab):
    """Rows cut into as many slices as the step's size asks for, and into the fewest that a workspace may allow: the same tokens."""
    from nano_vllm_x_amd import ops

    g = torch.Generator(device="cuda").manual_seed(vocab + rows)
    lg = (2.5 * torch.randn((rows, vocab), generator=g, device="cuda")).to(torch.bfloat16)
    r = torch.arange(rows, device="cuda")
    T = torch.where(r % 7 == 3, 0.0, 0.4 + 0.2 * (r % 5).float())
    k, p, m = torch.where(r % 4 == 0, 20, vocab), torch.where(r % 3 == 0, 0.8, 1.0), torch.where(r % 11 == 0, 0.1, 0.0)
    fewest = torch.empty(rows * max(1, min(16, 512 // rows)), dtype=torch.int64, device="cuda")
    want = ops.sample(lg, T, k, p, m, 3, 5, ws=fewest).cpu()
    assert torch.equal(_draw(lg, T, k, p, m, 3), want) and torch.equal(want[T.cpu() == 0], lg.float().argmax(1).cpu()[T.cpu() == 0])


@pytest.mark.parametrize("vocab,seed,offset,k,p,m,ids", [
    (5000, 1, 1, 5000, 1.0, 0.0, [2005, 2011, 3374, 3597, 4493, 2771, 435, 1119]),
    (5000, 1, 1, 50, 0.9, 0.05, [4623, 4681, 1956, 240, 3846, 4392, 4938, 4541]),
    (5000, 77, 123456789012, 5000, 1.0, 0.0, [3733, 435, 3381, 359, 312, 323, 1034, 301]),
    (5000, 77, 123456789012, 50, 0.9, 0.05, [1840, 3151, 914, 2469, 2349, 323, 4173, 3011]),
    (32000, 1, 1, 32000, 1.0, 0.0, [7340, 14449, 21241, 26118, 4493, 8429, 8018, 24926]),
    (32000, 1, 1, 50, 0.9, 0.05, [7340, 30361, 19564, 23902, 13105, 24539, 28112, 27438]),
    (32000, 77, 123456789012, 32000, 1.0, 0.0, [20498, 10211, 7836, 18574, 11933, 28992, 17831, 26739]),
    (32000, 77, 123456789012, 50, 0.9, 0.05, [14924, 6910, 13022, 29956, 14635, 22521, 16004, 29944])])
def test_a_seed_draws_the_tokens_it_drew(vocab, seed, offset, k, p, m, ids):
    """Draws recorded while the noise was made with __logf and 32-bit products."""
    from nano_vllm_x_amd import ops

    i, r = torch.arange(vocab)[None], torch.arange(8)[:, None]
    lg = (((i * 7919 + r * 104729) % 1009).float() / 250.0).bfloat16().cuda()
    f = lambda v, d=torch.float32: torch.full((8,), v, device="cuda", dtype=d)
    assert ops.sample(lg, f(0.8), f(k, torch.int64), f(p), f(m), seed, offset).tolist() == ids
