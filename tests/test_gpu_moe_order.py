"""ops.moe_order against a stable sort: edges of 64 pairs, of a wave's turn of 512 and of the workgroup's of 8192, every number of bits of an expert's number, experts that do not exist."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts", [1, 2, 3, 4, 5, 8, 9, 16, 17, 32, 33, 63])
@pytest.mark.parametrize("pairs", [1, 63, 64, 65, 1023, 1025, 8191, 8192, 8193, 20000])
def test_order_is_a_stable_sort(experts, pairs):
    from nano_vllm_x_amd import ops

    gen = torch.Generator().manual_seed(experts * pairs)
    for lo, hi in ((0, experts), (-2, experts + 3), (experts - 1, experts)):      # all exist, some do not, all pairs of one
        idx = torch.randint(lo, hi, (pairs, 1), generator=gen, dtype=torch.int32)
        dst, counts = (t.cpu() for t in ops.moe_order(idx.cuda(), experts))
        real = (idx >= 0) & (idx < experts)
        order = torch.argsort(idx[real].long(), stable=True)
        want = torch.empty(order.numel(), dtype=torch.int64)
        want[order] = torch.arange(order.numel())
        assert torch.equal(dst[real], want)
        assert torch.equal(counts.long(), torch.bincount(idx[real].long(), minlength=experts))


@pytest.mark.parametrize("experts", [1, 4, 5, 6, 7])
@pytest.mark.parametrize("pairs", [16384, 16385, 65536, 70001])
def test_many_pairs_of_few_experts(experts, pairs):
    """Several turns of every wave, on both sides of the line between a ballot an expert and a ballot a bit."""
    test_order_is_a_stable_sort(experts, pairs)
