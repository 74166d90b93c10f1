"""The products of prefill steps by every tile that csrc/prefill_gemm.hip has for many rows: edges of tiles, several tiles a workgroup, rows apart."""
import pytest
import torch

pytestmark = pytest.mark.gpu

WIDE = {1: (256, 256), 2: (192, 256), 3: (128, 256), 4: (128, 128), 5: (64, 128)}      # NVX_PG_* of csrc/prefill_gemm.h
UNIT = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}      # a unit in the last place of 8 (11) bits, of the value at most


def _product(x, w, silu, tile):
    from nano_vllm_x_amd import _lib, ops

    m, n = x.shape[0], w.shape[0] // 2 if silu else w.shape[0]
    y = torch.full((m + 3, n), 7.0, dtype=x.dtype, device="cuda")        # rows behind the last are not touched
    fn = getattr(_lib.load(), "nvx_internal_prefill_gemm" + ("_f16" if x.dtype == torch.float16 else ""))
    _lib.check(fn(x.data_ptr(), x.stride(0), w.data_ptr(), y.data_ptr(), m, w.shape[0], x.shape[1], int(silu), tile, ops._stream()))
    assert bool((y[m:] == 7.0).all())
    return y[:m]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("silu", [False, True])
@pytest.mark.parametrize("m,n,k", [(1, 256, 256), (127, 512, 256), (129, 256, 512), (191, 256, 1024), (193, 768, 256), (257, 512, 768), (700, 1024, 2048),
                                   (5130, 2048, 256), (16500, 1024, 256)])
def test_tiles(dtype, silu, m, n, k):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    wide = torch.randn(m, k + 64, generator=gen, device="cuda").to(dtype)
    x, w = wide[:, 32:32 + k], (torch.randn(n, k, generator=gen, device="cuda") * k ** -0.5).to(dtype)
    p = x.double() @ w.double().t()
    # the sums: every one of k additions in float32 rounds by 2^-24 of at most the sum of magnitudes; then one rounding to the format, half a unit in the
    # last place (with SILU of both projections, of silu's value and of the result: four, through a function of slope < 1.1)
    size = x.double().abs() @ w.double().abs().t()
    err = k * 2.0 ** -24 * size + UNIT[dtype] / 2 * p.abs() + 2.0 ** -25
    if silu:
        g, u, eg, eu = p[:, :n // 2], p[:, n // 2:], err[:, :n // 2], err[:, n // 2:]
        s = g * torch.sigmoid(g)
        es = 1.1 * eg + UNIT[dtype] / 2 * (s.abs() + 1.1 * eg) + 2.0 ** -20 * s.abs() + 2.0 ** -25       # (2^-20: the exponential and the quotient in float32)
        p, err = s * u, es * (u.abs() + eu) + s.abs() * eu
        err = err + UNIT[dtype] / 2 * (p.abs() + err) + 2.0 ** -25
    first = None
    for tile, (_, tn) in WIDE.items():
        if n % tn:
            continue
        got = _product(x, w, silu, tile)
        assert bool(((got.double() - p).abs() <= err).all()), tile
        first = got if first is None else first
        assert torch.equal(got, first), tile          # one order of summation whatever the tile


def test_long_steps_take_silu_and_mul_into_the_product():
    from nano_vllm_x_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(4500, 1024, generator=gen, device="cuda").bfloat16()
    w = (torch.randn(6144, 1024, generator=gen, device="cuda") / 32).bfloat16()
    assert ops.gated_product_fits(x, w)
    assert torch.equal(ops.gated_product(x, w), ops.silu_mul(_product(x, w, False, 1)))
    for a, b in ((x[:, 1:], w[:, 1:]), (x.float(), w.float()), (x, w.half()), (x.t(), w), (x[:, :768], w[:, :768]), (x[:0], w), (x.cpu(), w.cpu()), (x[:, :1000], w[:, :1000])):
        assert not ops.gated_product_fits(a, b)
