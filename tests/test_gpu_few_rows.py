"""ops.few_rows_product (the projections of decode steps of models with per-sequence state) against float64, at the edges of its tiles and rules,
and layers.linear's choice between it and the library."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(rows, n, k, dtype, seed, pad=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, k + pad, generator=g).to(dtype).cuda()[:, :k]
    w = (torch.randn(n, k, generator=g) * k ** -0.5).to(dtype).cuda()
    return x, w, torch.randn(n, generator=g).to(dtype).cuda()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,k", [(16, 512), (48, 1024), (1024, 1536), (2048, 2560), (4112, 512), (4128, 1024), (12288, 512), (12304, 512), (1024, 6144)])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 32])
def test_few_rows_product(rows, n, k, dtype):
    from nano_vllm_x_amd import ops

    x, w, b = _case(rows, n, k, dtype, rows + n + k, pad=8 * (rows % 3))
    exact = x.double() @ w.double().T
    # float32 sums of k products: each of the k additions rounds by 2^-24 of a partial sum, which |x| |w| bounds; a 16-bit result rounds once more
    slack = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    half_ulp = 2.0 ** (-9 if dtype == torch.bfloat16 else -12) * 2
    with torch.inference_mode():
        f32 = ops.few_rows_product(x, w, f32=True)
        plain, biased = ops.few_rows_product(x, w), ops.few_rows_product(x, w, b)
    assert f32.dtype == torch.float32 and bool(((f32.double() - exact).abs() <= slack).all())
    for got, ref in ((plain, exact), (biased, exact + b.double())):
        assert got.dtype == dtype and bool(((got.double() - ref).abs() <= slack + half_ulp * (ref.abs() + slack) + 2.0 ** -25).all())


def test_a_row_s_result_does_not_depend_on_the_others():
    from nano_vllm_x_amd import ops

    x, w, b = _case(32, 1024, 2048, torch.bfloat16, 5)
    with torch.inference_mode():
        whole = ops.few_rows_product(x, w, b)
        for r in (0, 7, 16, 31):
            assert torch.equal(ops.few_rows_product(x[r:r + 1], w, b)[0], whole[r])


def test_what_the_kernel_does_not_take_goes_to_the_library():
    from nano_vllm_x_amd import ops
    from nano_vllm_x_amd.layers.linear import Linear

    for rows, n, k, dtype, why in ((33, 1024, 1024, torch.bfloat16, "rows"), (4, 1000, 1024, torch.bfloat16, "outputs"), (4, 1024, 768, torch.bfloat16, "columns"),
                                   (4, 1024, 1024, torch.float32, "format")):
        x, w, b = _case(rows, n, k, dtype, 3)
        m = Linear(k, n).cuda().to(dtype)
        with torch.inference_mode():
            m.weight.copy_(w)
            m.bias.copy_(b)
            assert not ops.few_rows_fits(x, m.weight, m.bias), why
            assert torch.equal(m(x), torch.nn.functional.linear(x, w, b)), why
    x, w, b = _case(4, 1024, 1024, torch.bfloat16, 4, pad=4)      # rows 8 bytes off a 16-byte boundary
    assert not ops.few_rows_fits(x, w)
    m = Linear(1024, 1024).cuda().bfloat16()
    y = m(torch.randn(2, 1024, device="cuda").bfloat16().requires_grad_())      # under autograd as torch's own
    y.float().sum().backward()
    assert m.weight.grad is not None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,ff,k", [(1, 16, 512), (16, 3072, 1024), (17, 48, 1536), (32, 6144, 512)])
def test_gated_product_equals_product_and_activation(rows, ff, k, dtype):
    """The activation reads the projections rounded to the format either way: the same bits."""
    from nano_vllm_x_amd import ops

    x, w, _ = _case(rows, 2 * ff, k, dtype, rows + ff)
    with torch.inference_mode():
        gu = ops.few_rows_product(x, w)
        assert torch.equal(ops.few_rows_glu(x, w, gelu=True), ops.gelu_glu(gu))
        assert torch.equal(ops.few_rows_glu(x, w, 0.7, 1.702, 1.0), ops.moe_glu(gu, 0.7, 1.702, 1.0))
        assert torch.equal(ops.few_rows_glu(x, w, float("inf"), 1.0, 0.0), ops.moe_glu(gu, float("inf"), 1.0, 0.0))
