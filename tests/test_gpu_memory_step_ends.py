"""mlstm and gla for steps of one token per sequence with their small projections, norm and gate in the launch, against the separate launches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (keys not a multiple of the rows in flight, one column piece, the widest heads; inputs of less than a wave's piece and of several pieces a wave; ranks
# at the ends of their range)
@pytest.mark.parametrize("fmt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("heads,dim,vdim,k_in,rank", [(8, 64, 128, 1024, 16), (3, 40, 24, 260, 4), (1, 256, 1024, 2048, 32), (2, 100, 4, 36, 28)])
@pytest.mark.parametrize("kind", ["mlstm", "gla"])
def test_one_launch_equals_the_separate_ones(kind, heads, dim, vdim, k_in, rank, fmt):
    """The projections' sums have the same order, the recurrence is the same code, the sum of a head's squares has another: float32 but for the end,
    so a result may lie one unit of the format away where the two sides fall on both sides of a border."""
    from nano_vllm_x_amd import ops

    n = 5
    g = torch.Generator().manual_seed(dim + vdim)
    rnd = lambda *s: torch.randn(*s, generator=g)
    hd, he = heads * dim, heads * vdim
    x = rnd(n, 2 * hd + 2 * he + 4).to(fmt).cuda()[:, :2 * hd + 2 * he]
    h = rnd(n, k_in + 4).to(fmt).cuda()[:, :k_in]
    lay = ops.StepLayout(n, n, torch.tensor([0, 3, 9, 0, 70]).cuda(), torch.tensor([4, 0, -1, 2, 1], dtype=torch.int32).cuda())
    mem, norm, peak = rnd(5, heads, dim, vdim).cuda(), rnd(5, heads, dim).cuda(), rnd(5, heads).cuda()
    at, res = (0, hd, 2 * hd), []
    w1 = (rnd(2 * heads if kind == "mlstm" else rank, k_in) * k_in ** -0.5).cuda()
    w2, bias = (rnd(hd, rank).cuda(), rnd(hd).cuda()) if kind == "gla" else (None, rnd(2 * heads).cuda())
    w = rnd(he if kind == "mlstm" else vdim).cuda()
    assert ops.memory_step_fits(lay, h, mem, w1, w2)
    for one in (True, False):
        m, nn, p = mem.clone(), norm.clone(), peak.clone()
        if kind == "mlstm":
            if one:
                y = ops.mlstm_step(x, at, 2 * hd + he, h, w1, bias, 15.0, w, 1e-5, m, nn, p, lay, heads, dim, vdim)
            else:
                o = ops.mlstm_scan(x, at, ops.skinny_proj(h, w1), bias, 15.0, m, nn, p, lay, heads, dim, vdim)
                y = ops.head_norm_gate(o, w, 1e-5, gate=x[:, 2 * hd + he:], kind="sigmoid")
        elif one:
            y = ops.gla_step(x, at, 2 * hd + he, h, w1, w2, bias, 1 / 16, w, 1e-5, m, lay, heads, dim, vdim, q_mul=dim ** -0.5)
        else:
            alpha = ops.skinny_proj(ops.skinny_proj(h, w1), w2, bias=bias, out_act="sigmoid_pow", power=1 / 16)
            o = ops.gla_scan(x, at, alpha, m, lay, heads, dim, vdim, q_mul=dim ** -0.5)
            y = ops.head_norm_gate(o, w, 1e-5, gate=x[:, 2 * hd + he:], kind="silu")
        res.append((y.float()[[0, 1, 3, 4]], m, nn, p, y[2]))
    for got, want in zip(res[0][1:4], res[1][1:4]):
        assert float((got - want).abs().max()) <= dim * 2.0 ** -22 * float(want.abs().max())
    assert int((res[0][4] != 0).sum()) == 0                                  # a padding row
    got, want = res[0][0], res[1][0]
    step = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 0.0}[fmt]
    # (float32: the read-out's dim products, magnitudes of its largest; 16 bits: one unit more)
    assert bool(((got - want).abs() <= step * want.abs() + dim * 2.0 ** -21 * float(want.abs().max())).all())


def test_what_it_is_not_built_for_takes_the_separate_launches():
    from nano_vllm_x_amd import ops

    lay = ops.StepLayout(1, 1, torch.zeros(1, dtype=torch.int64).cuda(), torch.zeros(1, dtype=torch.int32).cuda())
    h, mem = torch.zeros(1, 64).cuda().bfloat16(), lambda d, e: torch.zeros(1, 2, d, e).cuda()
    w = lambda r, k=64: torch.zeros(r, k).cuda()
    assert ops.memory_step_fits(lay, h, mem(64, 64), w(4)) and ops.memory_step_fits(lay, h, mem(512, 1024), w(4))
    assert not ops.memory_step_fits(lay, h, mem(64, 66), w(4)) and not ops.memory_step_fits(lay, h, mem(516, 64), w(4))
    assert not ops.memory_step_fits(lay, torch.zeros(1, 128).cuda().bfloat16()[:, 2:66], mem(64, 64), w(4))
    assert ops.memory_step_fits(lay, h, mem(64, 64), w(16), w(128, 16)) and not ops.memory_step_fits(lay, h, mem(260, 64), w(16), w(520, 16))
    assert not ops.memory_step_fits(lay, h, mem(64, 64), w(18), w(128, 18)) and not ops.memory_step_fits(lay, h, mem(64, 64), w(36), w(128, 36))
