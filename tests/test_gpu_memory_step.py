"""decay, gla and mlstm for steps of one token per sequence against the scan kernels."""
import pytest
import torch

from seq_drivers import step_layout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("heads,dim,vdim", [(2, 64, 128), (1, 128, 256), (3, 40, 24), (2, 512, 4), (1, 7, 1024), (2, 100, 96)])
@pytest.mark.parametrize("kind", ["decay", "gla", "mlstm"])
def test_single_tokens_equal_the_ragged_form(kind, heads, dim, vdim, fmt):
    """The step without token offsets against the same step as portions of one token, which takes the scan kernels: float32 either way, sums
    of dim products in another order."""
    from nano_vllm_x_amd import ops

    n = 5
    g = torch.Generator().manual_seed(dim + vdim)
    hd, he = heads * dim, heads * vdim
    x = torch.randn(n, 2 * hd + he, generator=g).to(fmt).cuda()
    pos, slots = [0, 3, 9, 0, 70], [4, 0, -1, 2, 1]
    step = ops.StepLayout(n, n, torch.tensor(pos, dtype=torch.int64).cuda(), torch.tensor(slots, dtype=torch.int32).cuda())
    ragged = step_layout(ops, [1] * n, pos, slots)
    rnd = lambda *s: torch.randn(*s, generator=g).cuda()
    mem, norm, peak = rnd(5, heads, dim, vdim), rnd(5, heads, dim), rnd(5, heads)
    decay, alpha, gates, bias = torch.rand(heads, generator=g).cuda(), torch.rand(n, hd, generator=g).cuda(), 3 * rnd(n, 2 * heads), rnd(2 * heads)
    res = []
    for lay in (step, ragged):
        m, nn, p = mem.clone(), norm.clone(), peak.clone()
        if kind == "decay":
            o = ops.decay_scan(x, (0, hd, 2 * hd), decay, m, lay, heads, dim, vdim, act="silu", k_mul=0.5)
        elif kind == "gla":
            o = ops.gla_scan(x, (0, hd, 2 * hd), alpha, m, lay, heads, dim, vdim, q_mul=dim ** -0.5)
        else:
            o = ops.mlstm_scan(x, (0, hd, 2 * hd), gates, bias, 15.0, m, nn, p, lay, heads, dim, vdim)
        live = [i for i, s in enumerate(slots) if s >= 0]
        res.append((o.view(n, -1)[live], m, nn, p))
    for got, want in zip(*res):
        assert float((got - want).abs().max()) <= dim * 2.0 ** -22 * float(want.abs().max())
