"""Products of few rows that form the residual sum and the norm in front of them, against the separate launches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,k,n,gelu", [(1, 1024, 256, False), (16, 1024, 272, False), (15, 1024, 512, True), (8, 1024, 3072, False), (3, 1024, 1056, True)])
@pytest.mark.parametrize("parts", ["y", "y strided", "add", "all"])
def test_one_launch_equals_the_separate_ones(parts, rows, k, n, gelu, fmt):
    """The stream's sums are the same bits (one order); the norm's sum of squares has another, so an entry of h may lie one unit of the format away; the product
    is the separate kernel's of that h, bit for bit."""
    from nano_vllm_x_amd import ops

    g = torch.Generator().manual_seed(rows + k)
    rnd = lambda *s: torch.randn(*s, generator=g).cuda()
    x, w_norm, w = rnd(rows, k), rnd(k), (rnd(n, k) * k ** -0.5).to(fmt)
    y = None if parts == "add" else (3 * rnd(rows, k + 8)).to(fmt)[:, :k]
    if parts == "y":
        y = y.contiguous()
    add, x_bias = (rnd(rows, k), rnd(k)) if parts in ("add", "all") else (None, None)
    bias = rnd(n).to(fmt) if parts == "all" and not gelu else None
    with torch.no_grad():
        assert ops.lead_rows_fit(x, y, add, x_bias, w_norm, w, bias, gelu)
        keep = x.clone()
        new, h, out = ops.few_rows_lead(x, y, add, x_bias, w_norm, 1e-5, w, bias, gelu)
        assert torch.equal(x, keep)
        want_h = ops.residual_norm(x, y, add=add, bias=x_bias, w=w_norm, eps=1e-5, dtype=fmt)
        assert torch.equal(new, x)
        unit = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[fmt]
        assert bool(((h.float() - want_h.float()).abs() <= unit * want_h.float().abs() + 2.0 ** -24).all())
        want = ops.few_rows_glu(h, w, gelu=True) if gelu else ops.few_rows_product(h, w, bias)
        assert torch.equal(out, want)


def test_what_it_is_not_built_for_takes_the_separate_launches():
    from nano_vllm_x_amd import ops

    z = lambda *s, t=torch.float32: torch.zeros(*s, dtype=t, device="cuda")
    b = torch.bfloat16
    w, w2, one = z(512, 1024, t=b), z(512, 2048, t=b), z(1024)
    with torch.no_grad():
        fit = lambda x, y=None, norm=one, w=w, **kw: ops.lead_rows_fit(x, y, None, None, norm, w, **kw)
        assert fit(z(16, 1024)) and fit(z(1, 1024), z(1, 1024, t=b))
        assert not fit(z(17, 1024)) and not fit(z(4, 2048), norm=z(2048), w=w2) and not fit(z(0, 1024))
        assert not fit(z(4, 1024), w=z(240, 1024, t=b)) and not fit(z(4, 1024), w=z(512, 1024)) and not fit(z(4, 512), norm=z(512), w=z(512, 512, t=b))
        assert not fit(z(4, 1024), z(4, 1028, t=b)[:, :1024]) and not fit(z(4, 1025)[:, 1:]) and not fit(z(4, 1024), bias=z(512, t=b), gelu=True)
    assert not fit(z(4, 1024))          # (gradients)
