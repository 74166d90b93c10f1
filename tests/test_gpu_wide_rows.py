"""The row kernels that move several elements a thread, at the edges of the sizes they take, against float64 on the CPU: sublayer
boundaries of a post-normed stream, head norms behind gates, and the preparation of queries, keys and values."""
import pytest
import torch

from oracle import gibavik_oracle as go

pytestmark = pytest.mark.gpu

# half an ulp of the stored format on values of a few units, and float32 sums in another order
STORED = {torch.float32: 2e-5, torch.bfloat16: 2.0 ** -6, torch.float16: 2.0 ** -9}


@pytest.mark.parametrize("fmt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("width", [4, 1020, 1024, 1028, 2048, 2052, 4096, 4100])
def test_postnormed_boundary(fmt, width):
    from nano_vllm_x_amd import ops
    g = torch.Generator().manual_seed(width)
    t = 3
    x, wide = torch.randn(t, width, generator=g), torch.randn(t, 2 * width + 8, generator=g).to(fmt)
    y, y2 = wide[:, 4:4 + width], wide[:, 8 + width:]                     # rows of wider results
    per, nxt, one = torch.randn(width, generator=g), torch.randn(width, generator=g), torch.tensor([0.3, 1.7])[1:]
    cut = wide.cuda()
    got_x = x.cuda()
    h = ops.postnorm_residual(got_x, y=cut[:, 4:4 + width], y2=cut[:, 8 + width:], a=0.7, b=-1.3, w_post=per.cuda(), eps=1e-3, w_next=nxt.cuda())
    want = x.double() + go.unit_rms(0.7 * y.double() - 1.3 * y2.double(), 1e-3) * per
    assert torch.allclose(got_x.cpu().double(), want, atol=2e-5)
    assert torch.allclose(h.cpu().double(), go.unit_rms(want, 1e-3) * nxt, atol=STORED[fmt], rtol=STORED[fmt])
    # one number as the weight, standing off every border; the next sublayer reads the stream
    got_x = x.cuda()
    h = ops.postnorm_residual(got_x, y=cut[:, 4:4 + width], w_post=torch.tensor([0.3, 1.7]).cuda()[1:], eps=1e-3)
    want = x.double() + go.scalar_norm(y.double(), one, 1e-3)
    assert torch.allclose(got_x.cpu().double(), want, atol=2e-5) and torch.allclose(h.cpu().double(), want, atol=STORED[fmt], rtol=STORED[fmt])
    # the closing norm alone
    got_x = x.cuda()
    h = ops.postnorm_residual(got_x, w_next=nxt.cuda(), eps=1e-3, out_dtype=fmt)
    assert torch.equal(got_x.cpu(), x) and torch.allclose(h.cpu().double(), go.unit_rms(x.double(), 1e-3) * nxt, atol=STORED[fmt], rtol=STORED[fmt])
    # a result whose rows start off the border of four: element by element
    off = torch.randn(t, width + 1, generator=g).to(fmt)
    got_x = x.cuda()
    ops.postnorm_residual(got_x, y=off.cuda()[:, 1:], w_post=per.cuda(), eps=1e-3)
    assert torch.allclose(got_x.cpu().double(), x.double() + go.unit_rms(off[:, 1:].double(), 1e-3) * per, atol=2e-5)


@pytest.mark.parametrize("kind", ["none", "sigmoid", "silu"])
@pytest.mark.parametrize("heads,vdim", [(5, 64), (7, 128), (3, 256), (3, 252), (1, 508), (2, 512), (1, 1020), (1, 1028), (3, 2048), (1, 4096), (1, 4100)])
def test_head_norm_behind_a_gate(kind, heads, vdim):
    from nano_vllm_x_amd import ops
    g = torch.Generator().manual_seed(vdim)
    for t in (1, 5):
        o, w, z = torch.randn(t, heads, vdim, generator=g), torch.randn(heads * vdim, generator=g), torch.randn(t, heads * vdim + 12, generator=g)
        gate = {"none": 1.0, "sigmoid": torch.sigmoid(z.double()), "silu": z.double() * torch.sigmoid(z.double())}[kind]
        gate = gate if kind == "none" else gate[:, 4:4 + heads * vdim]
        for weight in (w, w[:vdim].contiguous(), None):
            got = ops.head_norm_gate(o.cuda(), None if weight is None else weight.cuda(), 1e-4, gate=z.cuda()[:, 4:4 + heads * vdim] if kind != "none" else None,
                                     kind=kind, dtype=torch.float32)
            scale = 1.0 if weight is None else weight.double().view(-1, vdim)
            want = (go.unit_rms(o.double(), 1e-4) * scale).reshape(t, -1) * gate
            assert torch.allclose(got.cpu().double().view(t, -1), want, atol=3e-5, rtol=1e-5)


@pytest.mark.parametrize("fmt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mode", ["head", "row", "none"])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("heads,kvh,dim,vdim,rot", [(16, 8, 128, 128, 64), (3, 1, 64, 64, 64), (5, 2, 128, 64, 16), (2, 1, 256, 128, 128), (3, 1, 64, 256, 32),
                                                    (32, 8, 128, 128, 128), (5, 3, 128, 128, 0), (3, 2, 128, 128, 96)])
def test_queries_keys_and_values_prepared(fmt, mode, interleaved, heads, kvh, dim, vdim, rot):
    """Pieces of eight elements: one head per part of a wave, whole and partial rotations; a value head that does not start on a border
    of its own size and a rotated part of 96 (whose halves are no power of two) take the element-wise kernel."""
    from nano_vllm_x_amd import ops
    from nano_vllm_x_amd.layers.rotary_embedding import rotary_frequencies
    g = torch.Generator().manual_seed(heads * dim + rot)
    t, base = 4, 3000.0
    nq, nk, nv = heads * dim, kvh * dim, kvh * vdim
    x = torch.randn(t, 8 + nq + nk + nv + 16, generator=g).to(fmt)
    pos, slots = torch.tensor([0, 1, 4095, 77]), torch.tensor([4, 0, -1, 6])
    qw, kw = (torch.randn(dim if mode == "head" else n, generator=g) for n in (nq, nk))
    freq = rotary_frequencies(rot, base)[0] if rot else None
    vfreq = rotary_frequencies(vdim, base)[0]
    xq, xk, xv = (u.double() for u in x[:, 8:8 + nq + nk + nv].split([nq, nk, nv], 1))
    if mode == "row":
        xq, xk = go.unit_rms(xq, 1e-4) * qw, go.unit_rms(xk, 1e-4) * kw
    xq, xk, xv = xq.reshape(t, heads, dim), xk.reshape(t, kvh, dim), xv.reshape(t, kvh, vdim)
    if mode == "head":
        xq, xk = go.unit_rms(xq, 1e-4) * qw, go.unit_rms(xk, 1e-4) * kw
    if rot:
        xq, xk = go.turn(xq, pos, base, rot, interleaved), go.turn(xk, pos, base, rot, interleaved)
    keep = slots >= 0
    for vf in (vfreq, None):
        kc, vc = torch.full((8, nk), 9.0, dtype=fmt).cuda(), torch.full((8, nv), 9.0, dtype=fmt).cuda()
        q, _ = ops.attn_prep_store(x.cuda(), (8, 8 + nq, 8 + nq + nk), pos.cuda(), qw.cuda(), kw.cuda(), mode, 1e-4, None if freq is None else freq.cuda(), rot,
                                   interleaved, None if vf is None else vf.cuda(), slots.cuda(), kc, vc, heads, kvh, dim, vdim)
        wv = xv if vf is None else go.turn(xv, pos, base, vdim, interleaved)
        for got, want in ((q, xq), (kc[slots[keep].cuda()], xk[keep]), (vc[slots[keep].cuda()], wv[keep])):
            assert torch.allclose(got.cpu().double(), want.reshape(got.shape), atol=STORED[fmt], rtol=STORED[fmt])
        assert (kc.cpu()[[1, 2, 3, 5, 7]] == 9.0).all() and (vc.cpu()[[1, 2, 3, 5, 7]] == 9.0).all()
    alone, _ = ops.attn_prep_store(x.cuda(), (8, 0, 0), pos.cuda(), qw.cuda(), None, mode, 1e-4, None if freq is None else freq.cuda(), rot, interleaved, None, None,
                                   None, None, heads, 0, dim, vdim)
    assert torch.equal(alone, q)
