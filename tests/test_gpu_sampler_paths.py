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


def test_min_p_keeps_the_tokens_of_its_ratio():
    """Among logits 0, -1, -2, ... at temperature 1 the ratio of a probability to the largest is e^-i: min_p between e^-3 and e^-2 leaves three tokens."""
    lg = torch.full((64, 1024), -100.0, device="cuda", dtype=torch.bfloat16)
    lg[:, 100:108] = -torch.arange(8, device="cuda").to(torch.bfloat16)
    z = lambda v, d=torch.float32: torch.full((64,), v, device="cuda", dtype=d)
    seen = set()
    for seed in range(60):
        seen |= set(_draw(lg, z(1.0), z(1024, torch.int64), z(1.0), z(0.09), seed).tolist())
    assert seen == {100, 101, 102}      # (the rarest of the three is drawn with probability 0.09: 3840 draws miss it with 1e-157)
