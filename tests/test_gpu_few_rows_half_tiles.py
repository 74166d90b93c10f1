"""Products of few rows whose workgroups take eight rows of the weight, against those that take 16: the same sums in the same order, so the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (the fewest outputs, an odd number of pairs of tiles, the most that go by eight; one and several turns of K)
@pytest.mark.parametrize("fmt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 32])
@pytest.mark.parametrize("n,k", [(16, 512), (48, 1536), (2048, 2048), (2032, 512), (64, 6144)])
@torch.no_grad()
def test_rows_of_eight_and_of_sixteen(n, k, rows, fmt):
    from nano_vllm_x_amd import ops

    g = torch.Generator().manual_seed(n + k + rows)
    rnd = lambda *s: torch.randn(*s, generator=g)
    x = rnd(rows, k + 8).to(fmt).cuda()[:, :k]
    big = (rnd(4096, k) * k ** -0.5).to(fmt).cuda()      # 4096 outputs go by 16 with up to 32 rows of x
    bias = rnd(4096).to(fmt).cuda()
    for f32 in (False, True):
        for b in (None, bias):
            want = ops.few_rows_product(x, big, b, f32=f32)[:, :n]
            got = ops.few_rows_product(x, big[:n], None if b is None else b[:n], f32=f32)
            assert torch.equal(got, want)
    # [gate | up] of 2 n outputs against one of 4128 (its halves' first n rows are the same)
    m = n if n % 16 == 0 and 2 * n <= 4096 else 16
    wide = torch.cat([(rnd(2064, k) * k ** -0.5) for _ in range(2)]).to(fmt).cuda()
    narrow = torch.cat([wide[:m], wide[2064:2064 + m]])
    for gelu in (False, True):
        want = ops.few_rows_glu(x, wide, 7.0, 1.702, 1.0, gelu)[:, :m]
        assert torch.equal(ops.few_rows_glu(x, narrow, 7.0, 1.702, 1.0, gelu), want)
