"""Experts of steps of many tokens as grouped products (ops.moe_expert_rows above 64 tokens in 16-bit formats) against float64: edges of the
128-pair tiles, experts that get none, one or all of the pairs, weights on the inputs and on the outputs, and a replayed capture."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def make(t, top, experts, width, ff, fmt, choose, seed):
    g = torch.Generator().manual_seed(seed)
    h, wts = torch.randn(t, width + 8, generator=g).to(fmt)[:, :width], torch.rand(t, top, generator=g) + 0.2
    w_gu, w_d = (torch.randn(*s, generator=g) * s[-1] ** -0.5 for s in ((experts, 2 * ff, width), (experts, width, ff)))
    idx = torch.stack([torch.randperm(choose, generator=g)[:top] for _ in range(t)]).to(torch.int32) + (experts - choose)
    return h, idx, wts, w_gu.to(fmt), w_d.to(fmt)


def expect(h, idx, wts, w_gu, w_d, limit, alpha, shift, weight_out):
    out = torch.zeros(h.shape, dtype=torch.float64)
    ff = w_d.shape[2]
    for e in range(w_gu.shape[0]):
        rows, k = (idx == e).nonzero(as_tuple=True)
        if rows.numel():
            s = wts[rows, k].double()[:, None]
            z = (h[rows].double() * (1.0 if weight_out else s)) @ w_gu[e].double().t()
            g, u = z[:, :ff].clamp(max=limit), z[:, ff:].clamp(-limit, limit)
            out.index_add_(0, rows, (g * torch.sigmoid(alpha * g) * (u + shift)) @ w_d[e].double().t() * (s if weight_out else 1.0))
    return out


@pytest.mark.parametrize("fmt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("t,top,experts,choose,width,ff", [(65, 1, 1, 1, 128, 64), (65, 2, 8, 8, 256, 192), (128, 1, 3, 1, 128, 64), (129, 1, 3, 2, 384, 128),
                                                           (300, 3, 63, 63, 128, 64), (1100, 2, 8, 5, 1024, 576), (2300, 2, 2, 2, 128, 64)])
@pytest.mark.parametrize("weight_out", [True, False])
def test_grouped_experts(fmt, t, top, experts, choose, width, ff, weight_out):
    from nano_vllm_x_amd import ops
    h, idx, wts, w_gu, w_d = make(t, top, experts, width, ff, fmt, choose, t + experts)
    args = (0.9, 1.702, 1.0) if weight_out else (float("inf"), 1.0, 0.0)
    dev = [x.cuda() for x in (h, idx, wts, w_gu, w_d)]
    got = ops.moe_expert_rows(*dev, *args, weight_out).cpu().double()
    want = expect(h, idx, wts, w_gu, w_d, *args, weight_out)
    # the hidden rows and the result are rounded to the format once each; sums are float32
    ulp = 2.0 ** -8 if fmt == torch.bfloat16 else 2.0 ** -11
    err = (got - want).abs()
    assert (err <= 2 * ulp * want.abs() + 4 * ulp * want.pow(2).mean().sqrt()).all(), (err / want.pow(2).mean().sqrt()).max()


def test_grouped_experts_in_a_replayed_graph():
    """The choices are read on the device: a capture replayed with other choices gives theirs."""
    from nano_vllm_x_amd import ops
    t, experts = 200, 8
    h, idx, wts, w_gu, w_d = (x.cuda() for x in make(t, 2, experts, 256, 64, torch.bfloat16, experts, 1))
    run = lambda: ops.moe_expert_rows(h, idx, wts, w_gu, w_d, float("inf"), 1.0, 0.0, True)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()
    for seed in (2, 3, 4):
        other = make(t, 2, experts, 256, 64, torch.bfloat16, 3 + seed % 3, seed)
        h.copy_(other[0])
        idx.copy_(other[1])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, run())
