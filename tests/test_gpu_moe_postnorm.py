"""The mixture whose sums of a token's choices are made in the launch of the norm behind them, against the separate launches: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (one, an odd number and several pairs a token; rows of one, two and four pieces a thread and of no whole number of them; experts streamed for few
# tokens, grouped, and both without a launch for the sums: float32, rows off the matrix tiles, a stream off its borders)
@pytest.mark.parametrize("fmt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("t,top,experts,width,ff", [(1, 2, 8, 2048, 64), (16, 1, 4, 1000, 40), (33, 3, 5, 4096, 64), (64, 2, 8, 1032, 24), (70, 2, 8, 4224, 64),
                                                    (65, 2, 4, 128, 64), (300, 3, 7, 1152, 128), (1100, 2, 8, 2176, 64), (3, 2, 4, 36, 6)])
@pytest.mark.parametrize("off", [False, True])
def test_same_bits(fmt, t, top, experts, width, ff, off):
    from nano_vllm_x_amd import ops

    g = torch.Generator().manual_seed(t + width)
    rnd = lambda *s: torch.randn(*s, generator=g)
    h, wts = rnd(t, width + 8).to(fmt).cuda()[:, :width], (torch.rand(t, top, generator=g) + 0.2).cuda()
    w_gu, w_d = (rnd(experts, 2 * ff, width) * width ** -0.5).to(fmt).cuda(), (rnd(experts, width, ff) * ff ** -0.5).to(fmt).cuda()
    idx = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(t)]).to(torch.int32).cuda()
    x0 = rnd(t * width + 1).cuda()[int(off):t * width + int(off)].view(t, width)
    for k, (weight_out, w_post, w_next, decode) in enumerate([(True, rnd(1), rnd(1), False), (True, rnd(width), None, True), (False, rnd(1), rnd(width), True)]):
        w_post, w_next = w_post.cuda(), w_next.cuda() if w_next is not None else None
        if k == 1:
            h[t // 2, 3] = float("inf")      # (a token's own affair: its sums are not numbers, its neighbours' are what they were)
        # (copies keep where a stream stands)
        xs = [torch.empty(t * width + 1, device="cuda")[int(off):t * width + int(off)].view(t, width).copy_(x0) for _ in range(2)]
        y = ops.moe_expert_rows(h, idx, wts, w_gu, w_d, float("inf"), 1.0, 0.0, weight_out, decode)
        want = ops.postnorm_residual(xs[0], y=y, w_post=w_post, eps=1e-5, w_next=w_next)
        got = ops.moe_expert_rows_postnorm(h, idx, wts, w_gu, w_d, float("inf"), 1.0, xs[1], w_post, 1e-5, 0.0, weight_out, decode, w_next)
        bits = lambda a: a.view(torch.int32 if a.dtype == torch.float32 else torch.int16)
        nan = want.isnan()
        assert torch.equal(nan, got.isnan()) and torch.equal(bits(want)[~nan], bits(got)[~nan])
        nan = xs[0].isnan()
        assert torch.equal(nan, xs[1].isnan()) and torch.equal(bits(xs[0].contiguous())[~nan], bits(xs[1].contiguous())[~nan])
        assert not want[:t // 2].isnan().any()
