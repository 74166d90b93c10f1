"""Attention of prompts by each form of the kernel whose tiles are fetched by waves of their own (32 positions of two heads as two waves, 64 of two, 32 of four): scores that climb
from tile to tile, scores that are infinite or no numbers, and tiles that a wave sees nothing of, against the loop without such waves and against float64."""
import pytest
import torch

from test_gpu_prefill_loaders import _against_float64, _run

pytestmark = pytest.mark.gpu
# query heads, key heads, sequences behind the first: blocks of 32 positions past one a CU take those of 64
FORMS = {"2 x 32": (4, 2, ()), "2 x 64": (4, 2, ((1400, 1400),) * 3), "4 x 32": (8, 2, ())}
MANY = ((64, 64),) * 400           # so many workgroups that no form has such waves


def _has_loaders(parts, hq, hkv, dtype):
    from nano_vllm_x_amd import _lib

    fn = getattr(_lib.load(), "nvx_internal_prefill_loaders" + ("_f16" if dtype == torch.float16 else ""))
    return bool(fn(sum(a for a, _ in parts), len(parts), hq, hkv))


def _inputs(part, form, dtype, seed):
    hq, hkv, more = FORMS[form]
    parts = (part, *more)
    assert _has_loaders(parts, hq, hkv, dtype) and not _has_loaders(parts + MANY, hq, hkv, dtype)
    # (of 32 positions of two heads as two waves up to 256 workgroups)
    assert ((sum(a for a, _ in parts) + 31) // 32 + len(parts) - 1) * hkv > 256 or form != "2 x 64"
    gen = torch.Generator(device="cuda").manual_seed(seed)
    nq, nk = (sum(p[i] for p in parts + MANY) for i in (0, 1))
    q = torch.randn(nq, hq, 128, generator=gen, device="cuda")
    k, v = (torch.randn(nk, hkv, 128, generator=gen, device="cuda") for _ in range(2))
    return hq, hkv, parts, q, k, v


def _both(q, k, v, parts, hq, hkv):
    """The launch with such waves, and the same rows of the one without."""
    n, slots = sum(a for a, _ in parts), torch.arange(k.shape[0], device="cuda", dtype=torch.int32)
    return _run(q[:n], k, v, parts, slots, hq, hkv), _run(q, k, v, parts + MANY, slots, hq, hkv)[:n], slots


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("part", [(150, 700), (321, 321), (65, 1000)])      # 321: a block's second wave ends a tile before the first one's last
@pytest.mark.parametrize("step", [0.25, 3.0, 5.5, 12.0, -3.0])
def test_scores_that_climb(dtype, form, part, step):
    hq, hkv, parts, q, k, v = _inputs(part, form, dtype, 7)
    q *= 0.1
    q[:, :, 0] = 128 ** 0.5                                  # a score is a key's first element, and what the others add
    k *= 0.5
    k[:, :, 0] += (torch.arange(k.shape[0], device="cuda") % part[1] // 64 * step)[:, None]
    q, k, v = q.view(len(q), -1).to(dtype), k.to(dtype), v.to(dtype)
    here, loop, slots = _both(q, k, v, parts, hq, hkv)
    assert torch.equal(here, loop)
    _against_float64(here, q, k, v, slots, part, hq, hkv, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", FORMS)
def test_the_largest_weight_is_exact(dtype, form):
    """Weights are taken relative to the largest score so far, whose weight is 1 in any format: where one key has nearly all of it and the rows of values are alike, a query gets that row, with no
    rounding of its weight in it (relative to an earlier, smaller score the weight itself is rounded, by up to half a unit, and so is the result)."""
    part = (64, 448)
    hq, hkv, parts, q, k, v = _inputs(part, form, dtype, 3)
    q.zero_()
    q[:, :, 0] = 128 ** 0.5 * torch.linspace(0.5, 1.0, len(q), device="cuda")[torch.randperm(len(q), generator=torch.Generator().manual_seed(1)).cuda()][:, None]
    k.zero_()
    k[:part[1], :, 0] = -40.0
    k[0, :, 0] = 0.0                                         # the largest of the first tile; the one behind exceeds it by 2^3.9 to 2^7.8
    k[330, :, 0] = 5.4
    unit = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    v[:] = 2.0 - unit                                        # (an error of half a unit of a weight is a whole one here)
    q, k, v = q.view(len(q), -1).to(dtype), k.to(dtype), v.to(dtype)
    here, loop, _ = _both(q, k, v, parts, hq, hkv)
    assert bool((here[:part[0]] == 2.0 - unit).all()) and bool((loop[:part[0]] == 2.0 - unit).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("part", [(1, 1), (1, 32), (1, 33), (1, 64), (1, 65), (33, 97), (1, 128), (64, 128), (1, 129), (64, 192), (1, 193), (64, 256), (1, 257), (64, 320), (64, 321), (1, 449)])
def test_few_tiles(dtype, form, part):
    """Up to four tiles are made one after the other, more by turns: edges of tiles and of their halves."""
    hq, hkv, parts, q, k, v = _inputs(part, form, dtype, sum(part))
    q, k, v = q.view(len(q), -1).to(dtype), k.to(dtype), v.to(dtype)
    here, loop, slots = _both(q, k, v, parts, hq, hkv)
    assert torch.equal(here, loop)
    _against_float64(here, q, k, v, slots, part, hq, hkv, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("key", [0, 63, 64, 300, 699])
def test_scores_that_are_no_numbers(dtype, form, value, key):
    """One element of one key: queries that do not see it have the bits that they have without it, the others what the loop makes of it."""
    part = (200, 700)
    hq, hkv, parts, q, k, v = _inputs(part, form, dtype, key)
    q[:, :, 5] = q[:, :, 5].abs() + 0.5                      # the score is of the value's sign
    q, k, v = q.view(len(q), -1).to(dtype), k.to(dtype), v.to(dtype)
    clean = _both(q, k, v, parts, hq, hkv)[0]
    k[key, :, 5] = value
    here, loop, _ = _both(q, k, v, parts, hq, hkv)
    assert torch.equal(here.isnan(), loop.isnan()) and torch.equal(here.nan_to_num(0.0), loop.nan_to_num(0.0))
    sees = torch.arange(part[0], device="cuda") + part[1] - part[0] >= key
    assert torch.equal(here[:part[0]][~sees], clean[:part[0]][~sees])
    if value == float("-inf"):
        assert bool(here.isfinite().all())                   # (weight 0; there are other keys)
    else:
        assert bool(here[:part[0]][sees].isnan().all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("part", [(150, 100), (300, 70), (130, 1), (200, 136)])
def test_waves_that_see_no_key(dtype, form, part):
    """Fewer keys than queries: the first queries see none and get zeros, and whole waves' first tile is hidden."""
    hq, hkv, parts, q, k, v = _inputs(part, form, dtype, sum(part))
    q, k, v = q.view(len(q), -1).to(dtype), k.to(dtype), v.to(dtype)
    here, loop, slots = _both(q, k, v, parts, hq, hkv)
    assert torch.equal(here, loop)
    blind = part[0] - part[1]
    assert bool((here[:blind] == 0).all())
    _against_float64(here[blind:], q[blind:], k, v, slots, (part[1], part[1]), hq, hkv, dtype)
