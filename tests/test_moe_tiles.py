"""Which tile the grouped products of experts take (the rule of csrc/moe_gemm.hip; no GPU: only the choice)."""
import pytest

from nano_vllm_x_amd import _lib

T256, T192, T128, FOUR_WAVES = 1, 2, 3, 4


@pytest.mark.parametrize("pairs,experts,n,k,tile", [
    (8192, 8, 3072, 1024, T256), (8192, 8, 1024, 1536, T192),           # two choices of 4096 tokens over experts of 1536 x 1024
    (130, 8, 3072, 1024, T128), (2200, 8, 3072, 1024, T192)])
def test_the_tile_of_the_fewest_rounds(pairs, experts, n, k, tile):
    assert _lib.load().nvx_internal_moe_tile(pairs, experts, n, k) == tile


@pytest.mark.parametrize("pairs,experts,n,k,slower", [
    (3200, 8, 3072, 1024, T192), (3200, 8, 6144, 2048, T192), (4400, 8, 3072, 1024, T256), (12000, 60, 2048, 512, T192), (16384, 60, 2048, 512, T256),
    (4400, 63, 1024, 1024, T192), (3200, 16, 2048, 1024, T192), (3200, 16, 1024, 1024, T128), (8000, 8, 512, 256, T128), (260, 63, 1024, 1024, T128)])
def test_no_tile_that_counts_make_slower_than_the_kernel_of_four_waves(pairs, experts, n, k, slower):
    """(Measured: the tile costs 3 to 20 % of the mixture there.)"""
    assert _lib.load().nvx_internal_moe_tile(pairs, experts, n, k) != slower


def test_products_that_the_wide_tiles_do_not_read():
    for pairs in (65, 1000, 100000):
        assert _lib.load().nvx_internal_moe_tile(pairs, 8, 1024, 192) == FOUR_WAVES      # fewer steps of columns than they have on their way
        assert _lib.load().nvx_internal_moe_tile(pairs, 8, 1152, 1024) in (T128, FOUR_WAVES)
