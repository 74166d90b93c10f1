"""The tile of 96 x 64 of csrc/prefill_gemm.hip: edges of tiles, one and several rounds of workgroups, rows apart, against the tile of 64 x 64 (held to float64 elsewhere)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(1, 128, 256), (95, 128, 256), (96, 256, 512), (97, 128, 768), (1025, 1024, 2048), (1100, 4096, 256), (1536, 1024, 256)])
def test_one_order_of_summation(dtype, m, n, k):
    from nano_vllm_x_amd import _lib, ops

    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k + 64, generator=gen, device="cuda").to(dtype)[:, 32:32 + k]
    w = (torch.randn(n, k, generator=gen, device="cuda") * k ** -0.5).to(dtype)
    fn, out = getattr(_lib.load(), "nvx_internal_prefill_gemm" + ("_f16" if dtype == torch.float16 else "")), []
    for tile in (6, 7, 0):       # 64 x 64, 96 x 64, by the rule
        y = torch.full((m, n), float("nan"), dtype=dtype, device="cuda")
        _lib.check(fn(x.data_ptr(), x.stride(0), w.data_ptr(), y.data_ptr(), m, n, k, 0, tile, ops._stream()))
        out.append(y)
    assert bool(torch.isfinite(out[0]).all()) and torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
    y = torch.empty((m, n // 2), dtype=dtype, device="cuda")
    with pytest.raises(RuntimeError):
        _lib.check(fn(x.data_ptr(), x.stride(0), w.data_ptr(), y.data_ptr(), m, n, k, 1, 7, ops._stream()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(1, 128, 256), (127, 128, 512), (129, 256, 768), (159, 128, 1024), (161, 128, 256), (193, 1024, 512), (320, 128, 1280), (577, 4096, 256), (2100, 1024, 3072)])
def test_tall_tiles_and_few_steps(dtype, m, n, k):
    """Tiles of 128, 160 and 192 x 64, and those of 32 rows whose steps of 128 columns are fewer than a ring holds: the bits of 64 x 64, no row past the last written."""
    from nano_vllm_x_amd import _lib, ops

    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k + 64, generator=gen, device="cuda").to(dtype)[:, 32:32 + k]
    w = (torch.randn(n, k, generator=gen, device="cuda") * k ** -0.5).to(dtype)
    fn, first = getattr(_lib.load(), "nvx_internal_prefill_gemm" + ("_f16" if dtype == torch.float16 else "")), None
    for tile in (6, 11, 12, 13, 5, 8, 9):
        y = torch.full((m + 200, n), float("nan"), dtype=dtype, device="cuda")
        _lib.check(fn(x.data_ptr(), x.stride(0), w.data_ptr(), y.data_ptr(), m, n, k, 0, tile, ops._stream()))
        first = y[:m] if first is None else first
        assert bool(torch.isfinite(y[:m]).all()) and bool(torch.isnan(y[m:]).all()) and torch.equal(y[:m], first), tile
    for tile in (9, 11, 12, 13):      # no SiluAndMul in these
        with pytest.raises(RuntimeError):
            _lib.check(fn(x.data_ptr(), x.stride(0), w.data_ptr(), y.data_ptr(), m, n, k, 1, tile, ops._stream()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(1, 128, 256), (63, 256, 512), (65, 128, 768), (95, 128, 1024), (97, 256, 256), (159, 128, 1280), (161, 256, 512), (193, 384, 256), (223, 128, 512),
                                   (225, 128, 256), (449, 1024, 1024), (768, 6144, 1024), (1024, 6144, 256)])
def test_tiles_as_wide_as_128(dtype, m, n, k):
    """Tiles of 64, 96, 160, 192 and 224 x 128, plain and with SiluAndMul: the bits of 64 x 64, no row past the last written."""
    from nano_vllm_x_amd import _lib, ops

    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k + 64, generator=gen, device="cuda").to(dtype)[:, 32:32 + k]
    w = (torch.randn(n, k, generator=gen, device="cuda") * k ** -0.5).to(dtype)
    fn = getattr(_lib.load(), "nvx_internal_prefill_gemm" + ("_f16" if dtype == torch.float16 else ""))
    for silu in (0, 1):
        first = None
        for tile in (6, 5, 14, 16, 17, 18, 0):
            y = torch.full((m + 230, n // (1 + silu)), float("nan"), dtype=dtype, device="cuda")
            _lib.check(fn(x.data_ptr(), x.stride(0), w.data_ptr(), y.data_ptr(), m, n, k, silu, tile, ops._stream()))
            first = y[:m] if first is None else first
            assert bool(torch.isfinite(y[:m]).all()) and bool(torch.isnan(y[m:]).all()) and torch.equal(y[:m], first), (silu, tile)
        for tile in (10, 15, 19):      # heads' tiles and none
            with pytest.raises(RuntimeError):
                _lib.check(fn(x.data_ptr(), x.stride(0), w.data_ptr(), y.data_ptr(), m, n, k, silu, tile, ops._stream()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(1, 128, 256), (63, 256, 512), (64, 128, 768), (65, 384, 1024), (129, 256, 1280), (1030, 6144, 256), (4096, 1536, 256), (2049, 3072, 512)])
def test_three_workgroups_a_cu(dtype, m, n, k):
    """SiluAndMul by 64 x 128 with two steps in LDS, and by the rule's tile: the bits of 64 x 64, no row past the last written; no plain product in it."""
    from nano_vllm_x_amd import _lib, ops

    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k + 64, generator=gen, device="cuda").to(dtype)[:, 32:32 + k]
    w = (torch.randn(n, k, generator=gen, device="cuda") * k ** -0.5).to(dtype)
    fn, first = getattr(_lib.load(), "nvx_internal_prefill_gemm" + ("_f16" if dtype == torch.float16 else "")), None
    for tile in (6, 20, 0):
        y = torch.full((m + 70, n // 2), float("nan"), dtype=dtype, device="cuda")
        _lib.check(fn(x.data_ptr(), x.stride(0), w.data_ptr(), y.data_ptr(), m, n, k, 1, tile, ops._stream()))
        first = y[:m] if first is None else first
        assert bool(torch.isfinite(y[:m]).all()) and bool(torch.isnan(y[m:]).all()) and torch.equal(y[:m], first), tile
    y = torch.empty((m, n), dtype=dtype, device="cuda")
    with pytest.raises(RuntimeError):
        _lib.check(fn(x.data_ptr(), x.stride(0), w.data_ptr(), y.data_ptr(), m, n, k, 0, 20, ops._stream()))
