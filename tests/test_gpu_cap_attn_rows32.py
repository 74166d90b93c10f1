"""ops.softcap_attn for heads of 128 on the matrix cores (tiles of 64 keys shared by four waves) against float64: head groups of one, two and four,
edges of the 32-query and 64-key blocks, continued portions, windows with kept first keys, chunks, caps, penalties, sinks, tied keys and
values, read-outs turned back and gated, and steps of more sequences than a wave has lanes."""
import math

import numpy as np
import pytest
import torch

from seq_drivers import step_layout

pytestmark = pytest.mark.gpu
F64 = torch.float64


def case(lens, totals, heads, kvh, fmt, seed):
    g = torch.Generator().manual_seed(seed)
    n = sum(totals)
    perm = torch.randperm(n, generator=g)
    slots = [perm[sum(totals[:b]):sum(totals[:b + 1])] for b in range(len(totals))]
    rows = lambda r, c: torch.randn(r, c, generator=g).to(fmt)
    return rows(sum(lens), heads * 128), rows(n, kvh * 128), rows(n, kvh * 128), slots, g


def call(ops, lens, totals, q, k, v, slots, heads, kvh, softcap=0.0, **kw):
    lay = step_layout(ops, lens, [n - l for n, l in zip(totals, lens)], list(range(len(lens))))
    start = torch.tensor(np.concatenate([[0], np.cumsum(totals)[:-1]]), dtype=torch.int64).cuda()
    kc = k.cuda()
    return ops.softcap_attn(q.cuda(), kc, kc if v is k else v.cuda(), torch.cat(slots).to(torch.int32).cuda(), start,
                            torch.tensor(totals, dtype=torch.int32).cuda(), lay, cap=softcap, heads=heads, kv_heads=kvh, dim=128, vdim=128, **kw)


def expect(lens, totals, q, k, v, slots, heads, kvh, scale, softcap=0.0, window=0, chunk=0, keep=0, r1=None, r2=None, slopes=None, sinks=None, k_rn=None):
    out, at, g = [], 0, heads // kvh
    for l, n, s in zip(lens, totals, slots):
        qs, ks, vs = q[at:at + l].double().view(l, heads, 128), k[s].double().view(n, kvh, 128), v[s].double().view(n, kvh, 128)
        if k_rn is not None:
            ks = ks * k_rn[s].double()[..., None]
        i, j = torch.arange(n - l, n)[:, None], torch.arange(n)[None]
        far = i - j
        seen = far >= 0
        if window:
            seen = seen & ((far < window) | (j < keep))
        if chunk:
            seen = seen & (i // chunk == j // chunk)
        z = torch.einsum("ihd,jhd->hij", qs, ks.repeat_interleave(g, 1)) * scale
        if softcap:
            z = softcap * torch.tanh(z / softcap)
        if r1 is not None:
            z = z - r1.double()[:, None, None] * torch.log1p(r2.double()[:, None, None] * far.clamp(min=0))
        if slopes is not None:
            z = z - slopes.double()[:, None, None] * far
        z = z.masked_fill(~seen, -math.inf)
        if sinks is not None:
            z = torch.cat([z, sinks.double()[:, None, None].expand(heads, l, 1)], 2)
        p = torch.softmax(z, 2)[..., :n]
        out.append(torch.einsum("hij,jhd->ihd", p, vs.repeat_interleave(g, 1)).reshape(l, -1))
        at += l
    return torch.cat(out)


def near(got, want, fmt):
    ulp = 2.0 ** -8 if fmt == torch.bfloat16 else 2.0 ** -11       # one rounding of the result; weights keep 16 bits, sums are float32
    err = (got.cpu().double() - want).abs()
    assert (err <= ulp * want.abs() + 1e-4).all(), err.max()


LENS = ([1, 31, 33, 64, 65, 200], [1, 64, 100, 64, 193, 331])        # tokens of the step, and of the sequence


@pytest.mark.parametrize("heads,kvh", [(4, 4), (6, 3), (8, 2), (12, 2)])
@pytest.mark.parametrize("fmt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["plain", "window", "kept", "chunk", "cap", "log", "slopes", "sinks"])
def test_head_groups_and_masks(heads, kvh, fmt, kind):
    from nano_vllm_x_amd import ops
    q, k, v, slots, g = case(*LENS, heads, kvh, fmt, heads)
    per_head = lambda: torch.rand(heads, generator=g) + 0.1
    kw = {"plain": {}, "window": {"window": 70}, "kept": {"window": 40, "keep": 67}, "chunk": {"chunk": 50}, "cap": {"softcap": 3.0},
          "log": {"r1": per_head(), "r2": per_head()}, "slopes": {"slopes": per_head()}, "sinks": {"sinks": 4.0 * per_head()}}[kind]
    dev = {a.replace("keep", "keep_first"): b.cuda() if isinstance(b, torch.Tensor) else b for a, b in kw.items() if a != "softcap"}
    got = call(ops, *LENS, q, k, v, slots, heads, kvh, scale=0.11, softcap=kw.get("softcap", 0.0), **dev)
    near(got, expect(*LENS, q, k, v, slots, heads, kvh, 0.11, **kw), fmt)


@pytest.mark.parametrize("chunk", [0, 64, 100])
@pytest.mark.parametrize("heads,kvh", [(2, 2), (4, 2), (4, 1)])
def test_tied_keys_and_values(chunk, heads, kvh):
    from nano_vllm_x_amd import ops
    q, k, _, slots, g = case(*LENS, heads, kvh, torch.bfloat16, 3)
    rn, slopes = torch.rand(k.shape[0], kvh, generator=g) + 0.5, torch.rand(heads, generator=g)
    got = call(ops, *LENS, q, k, k, slots, heads, kvh, scale=0.09, chunk=chunk, slopes=slopes.cuda(), k_rn=rn.cuda())
    near(got, expect(*LENS, q, k, k, slots, heads, kvh, 0.09, chunk=chunk, slopes=slopes, k_rn=rn), torch.bfloat16)


@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("per_head", [False, True])
def test_read_out_turned_back_and_gated(interleaved, per_head):
    from nano_vllm_x_amd import ops
    heads, kvh, fmt = 4, 2, torch.float16
    q, k, v, slots, g = case(*LENS, heads, kvh, fmt, 5)
    t = q.shape[0]
    ang = 6.0 * torch.rand(t, 64, generator=g)
    gate = torch.randn(t, heads if per_head else heads * 128 + 8, generator=g).to(fmt)
    cut = gate if per_head else gate[:, 8:]
    out = torch.zeros(t, heads * 128 + 16, dtype=fmt).cuda()
    call(ops, *LENS, q, k, v, slots, heads, kvh, scale=0.1, v_turn=torch.cat([ang.cos(), ang.sin()], 1).cuda(), v_interleaved=interleaved,
         gate=gate.cuda() if per_head else gate.cuda()[:, 8:], out_mul=1.5, out=out[:, 8:8 + heads * 128])
    o = 1.5 * expect(*LENS, q, k, v, slots, heads, kvh, 0.1).view(t, heads, 128)
    u, w = (o[..., 0::2], o[..., 1::2]) if interleaved else (o[..., :64], o[..., 64:])
    c, s = ang.cos().double()[:, None], ang.sin().double()[:, None]
    a, b = u * c + w * s, w * c - u * s
    o = torch.stack([a, b], -1).flatten(2) if interleaved else torch.cat([a, b], 2)
    z = torch.sigmoid(cut.double())
    near(out[:, 8:8 + heads * 128], (o * (z[..., None] if per_head else z.view(t, heads, 128))).reshape(t, -1), fmt)
    assert (out[:, :8] == 0).all() and (out[:, -8:] == 0).all()


@pytest.mark.parametrize("n_seq,longest", [(3, 700), (64, 130), (70, 130), (130, 40)])
def test_many_sequences(n_seq, longest):
    """Every block of every sequence is taken once, whatever order the workgroups take them in."""
    from nano_vllm_x_amd import ops
    g = torch.Generator().manual_seed(n_seq)
    lens = torch.randint(1, longest, (n_seq,), generator=g).tolist()
    q, k, v, slots, _ = case(lens, lens, 4, 2, torch.bfloat16, n_seq)
    near(call(ops, lens, lens, q, k, v, slots, 4, 2, scale=0.1), expect(lens, lens, q, k, v, slots, 4, 2, 0.1), torch.bfloat16)
