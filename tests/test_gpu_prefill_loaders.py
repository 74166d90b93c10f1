"""Attention of prompts in launches of few workgroups, whose tiles are fetched by waves of their own: the bits of the same sequences among many others."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(q, k, v, parts, slots, hq, hkv):
    """parts: (queries, keys) of each sequence, whose queries are the next rows of q and keys the next of the slot list."""
    from nano_vllm_x_amd import ops

    ends = torch.tensor([(0, 0)] + list(parts)).cumsum(0).to(torch.int32).cuda()
    qo, kv = ends[:, 0].contiguous(), ends[:, 1].contiguous()
    plan = ops.prefill_plan_ws(len(parts), "cuda")
    ops.prefill_plan(qo, plan)
    return ops.paged_prefill(q, k, v, qo, kv, slots, plan, hq, hkv, 128 ** -0.5)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv", [(4, 2), (8, 2)])
@pytest.mark.parametrize("parts", [((1, 1),), ((31, 31),), ((33, 64),), ((64, 65),), ((1, 128),), ((129, 129),), ((200, 700),), ((449, 449), (2, 300)), ((3, 3), (65, 1000), (1, 64), (640, 641)),
                                   ((1000, 1400), (500, 500), (300, 2000))])
def test_the_same_alone_and_among_others(dtype, hq, hkv, parts):
    gen = torch.Generator(device="cuda").manual_seed(sum(a + 7 * b for a, b in parts))
    filler = ((64, 64),) * 200           # so many workgroups that the copies are every wave's
    nq, nk = (sum(p[i] for p in parts + filler) for i in (0, 1))
    q = torch.randn(nq, hq * 128, generator=gen, device="cuda").to(dtype)
    k, v = (torch.randn(nk, hkv, 128, generator=gen, device="cuda").to(dtype) for _ in range(2))
    slots = torch.randperm(nk, generator=gen, device="cuda").to(torch.int32)
    n = sum(p[0] for p in parts)
    alone = _run(q[:n], k, v, parts, slots, hq, hkv)
    among = _run(q, k, v, parts + filler, slots, hq, hkv)
    assert bool(torch.isfinite(alone).all()) and torch.equal(alone, among[:n])
    _against_float64(alone, q, k, v, slots, parts[0], hq, hkv, dtype)


def _against_float64(got, q, k, v, slots, part, hq, hkv, dtype):
    """The first sequence of a launch."""
    (a, b), heads = part, hq // hkv
    rows = slots[:b].long()
    s = torch.einsum("ihd,jhd->hij", q[:a].view(a, hq, 128).double(), k[rows].double().repeat_interleave(heads, 1)) * 128 ** -0.5
    s = s.masked_fill(torch.arange(b, device="cuda")[None] > torch.arange(a, device="cuda")[:, None] + b - a, -torch.inf).softmax(2)
    want = torch.einsum("hij,jhd->ihd", s, v[rows].double().repeat_interleave(heads, 1)).reshape(a, -1)
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    size = torch.einsum("hij,jhd->ihd", s, v[rows].double().abs().repeat_interleave(heads, 1)).reshape(a, -1)
    # weights rounded to the format (half a unit each, the sum of them is not), the result once more; scores in float32
    assert bool(((got[:a].double() - want).abs() <= unit * size + unit * want.abs() + 2.0 ** -14 * size).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("step", [0.25, 3.0, 5.5, 12.0, -3.0])
def test_scores_that_climb(dtype, step):
    """Scores that rise by `step` from tile to tile (and fall): what weights are taken relative to moves with every tile, or stays."""
    gen = torch.Generator(device="cuda").manual_seed(7)
    part, filler, hq, hkv = (150, 700), ((64, 64),) * 200, 4, 2
    nq, nk = part[0] + 64 * 200, part[1] + 64 * 200
    q = torch.zeros(nq, hq, 128, device="cuda")
    q[:, :, 0] = 128 ** 0.5                                  # a score is a key's first element, and what the others add
    q[:, :, 1:] = 0.1 * torch.randn(nq, hq, 127, generator=gen, device="cuda")
    k = 0.5 * torch.randn(nk, hkv, 128, generator=gen, device="cuda")
    k[:, :, 0] += (torch.arange(nk, device="cuda") % part[1] // 64 * step)[:, None]
    q, k, v = q.view(nq, -1).to(dtype), k.to(dtype), torch.randn(nk, hkv, 128, generator=gen, device="cuda").to(dtype)
    slots = torch.arange(nk, device="cuda", dtype=torch.int32)
    alone = _run(q[:part[0]], k, v, (part,), slots, hq, hkv)
    assert torch.equal(alone, _run(q, k, v, (part, *filler), slots, hq, hkv)[:part[0]])
    _against_float64(alone, q, k, v, slots, part, hq, hkv, dtype)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 130])
def test_blocks_in_order_of_length(n):
    """Up to 64 sequences the longest blocks of all go first, more in the order of the sequences: every row is computed, empty sequences among them, and gives the bits it gives alone."""
    gen = torch.Generator(device="cuda").manual_seed(n)
    parts = [(0 if i % 7 == 3 else (17 * i * i + 5) % 210 + 1, 0) for i in range(n)]
    parts = [(a, a + (61 * i) % 400) for i, (a, _) in enumerate(parts)]
    nq, nk = (sum(p[i] for p in parts) for i in (0, 1))
    q = torch.randn(nq, 4 * 128, generator=gen, device="cuda").bfloat16()
    k, v = (torch.randn(nk, 2, 128, generator=gen, device="cuda").bfloat16() for _ in range(2))
    slots = torch.randperm(nk, generator=gen, device="cuda").to(torch.int32)
    got, at_q, at_k = _run(q, k, v, parts, slots, 4, 2), 0, 0
    for a, b in parts:
        if a:
            assert torch.equal(_run(q[at_q:at_q + a], k, v, [(a, b)], slots[at_k:at_k + b].clone(), 4, 2), got[at_q:at_q + a])
        at_q, at_k = at_q + a, at_k + b


@pytest.mark.parametrize("n", [63, 64, 65, 300])
def test_no_plan_is_read_where_none_is_made(n):
    """Through the wrapper, which makes a plan only for more sequences than the kernel says: with its workspace empty every row is there, and right."""
    from nano_vllm_x_amd import ops
    from nano_vllm_x_amd.layers.attention import PagedPrefillWrapper

    gen = torch.Generator(device="cuda").manual_seed(n)
    parts = [(i % 70, i % 70 + i % 11) for i in range(1, n + 1)]
    ends = torch.tensor([(0, 0)] + parts).cumsum(0).to(torch.int32).cuda()
    qo, kv = ends[:, 0].contiguous(), ends[:, 1].contiguous()
    nq, nk = int(qo[-1]), int(kv[-1])
    q = torch.randn(nq, 4 * 128, generator=gen, device="cuda").bfloat16()
    k, v = (torch.randn(nk, 2, 128, generator=gen, device="cuda").bfloat16() for _ in range(2))
    slots = torch.randperm(nk, generator=gen, device="cuda").to(torch.int32)
    w = PagedPrefillWrapper()
    w._plan_ws = ops.prefill_plan_ws(n, "cuda")
    w.plan(qo, kv, slots, None, 4, 2, 128)
    assert bool((w._plan_ws != 0).any()) == (n > ops.prefill_planless())
    out = torch.full((nq, 4 * 128), torch.nan, device="cuda", dtype=torch.bfloat16)
    assert torch.equal(w.run(q, (k, v), out=out).reshape(nq, -1), _run(q, k, v, parts, slots, 4, 2))
