"""Which launches of csrc/prefill_attn.hip have waves that only fetch (host code): every one of up to 392 workgroups, and up to 512 only where one or two sequences make them."""
import pytest


def _loaders(suffix, lens, hq, hkv):
    from nano_vllm_x_amd import _lib

    return bool(getattr(_lib.load(), "nvx_internal_prefill_loaders" + suffix)(sum(lens), len(lens), hq, hkv))


@pytest.mark.parametrize("suffix", ["", "_f16"])
def test_prompts_of_one_length(suffix):
    for lens in ([400] * 8, [452] * 8, [269] * 12, [194] * 16, [744] * 4, [602] * 6):         # 408 to 512 workgroups of 64 positions, slower with them by 0.4 to 3 %
        assert not _loaders(suffix, lens, 16, 8)
    for lens in ([237] * 6, [218] * 8, [134] * 12, [444] * 4, [968] * 2):                      # of 32 positions
        assert not _loaders(suffix, lens, 32, 8)


@pytest.mark.parametrize("suffix", ["", "_f16"])
def test_where_they_are_the_faster(suffix):
    for lens in ([459], [3168], [4064], [1552] * 2, [2000] * 2, [2638, 466], [340] * 6, [200] * 12, [100, 200, 300, 400, 500, 512]):
        assert _loaders(suffix, lens, 16, 8)
    for lens in ([459], [1500], [2000], [200] * 6):
        assert _loaders(suffix, lens, 32, 8)
    for lens, hq in (([4097], 16), ([2049] * 2, 16), ([2049], 32), ([459], 8), ([459], 64)):   # three rounds; other numbers of heads
        assert not _loaders(suffix, lens, hq, 8)
