"""The tile that csrc/prefill_gemm.hip's rule takes for a product (host code), at sizes where the tiles were timed and one is the best by far."""
import pytest

T64X128, T128, T192X256, THREE = 5, 4, 2, 20


@pytest.mark.parametrize("suffix", ["", "_f16"])
@pytest.mark.parametrize("m,n,k,tile", [
    # SiluAndMul of narrow layers: what a round costs however few its columns are (us by this tile / by the one that costs linear in the columns gave)
    (4096, 1536, 256, THREE), (2048, 3072, 256, THREE), (1836, 3072, 256, THREE),      # 8.1 / 12.4, 8.1 / 9.7, 8.0 / 9.5
    (3072, 3072, 256, T192X256), (1536, 6144, 256, T192X256),                          # 12.2 / 15.5, 12.5 / 15.9
    (2048, 3072, 512, THREE), (1024, 3072, 512, T128), (512, 6144, 512, T128),         # 12.3 / 13.2, 8.7 / 9.8, 9.0 / 10.3
    (2172, 4096, 512, T192X256), (4474, 4096, 512, T192X256),                          # 18.2 / 20.2, 31.8 / 34.1
    (1854, 4608, 768, T192X256), (2907, 3072, 768, T192X256),                          # 23.7 / 25.1, 22.8 / 24.1
    (256, 6144, 1024, T64X128)])
def test_silu_tiles(suffix, m, n, k, tile):
    from nano_vllm_x_amd import _lib

    assert getattr(_lib.load(), "nvx_internal_prefill_tile" + suffix)(m, n, k, 1) == tile


def test_three_a_cu_only_while_all_run_at_once():
    from nano_vllm_x_amd import _lib

    rule, taken = _lib.load().nvx_internal_prefill_tile, 0
    for k in (256, 512, 768, 1024, 2048):
        for n in (256, 1024, 1536, 3072, 6144, 12288):
            for m in range(1, 9000, 61):
                assert rule(m, n, k, 0) != THREE
                if rule(m, n, k, 1) == THREE:
                    taken += 1
                    assert -(-m // 64) * (n // 128) <= 768
    assert taken
