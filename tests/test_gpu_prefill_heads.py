"""Heads normed and turned at the end of the qkv product (csrc/prefill_gemm.hip): the bits of the plain product with nvx_qknorm_rope_store behind it, by every tile and by the rule's."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k,hq,hkv", [(1, 256, 2, 1), (31, 256, 4, 2), (32, 512, 16, 8), (33, 768, 2, 2), (63, 256, 4, 2), (65, 1024, 8, 4), (96, 256, 2, 1), (97, 512, 4, 1), (127, 1280, 2, 1),
                                        (129, 256, 4, 2), (257, 1024, 16, 8), (459, 1024, 16, 8), (700, 512, 16, 8), (1025, 256, 2, 1), (1500, 1024, 16, 8)])
def test_same_bits_as_a_launch_behind_the_product(dtype, m, k, hq, hkv):
    from nano_vllm_x_amd import _lib, ops

    gen = torch.Generator(device="cuda").manual_seed(m + k)

    def randn(*shape):
        return torch.randn(shape, generator=gen, device="cuda")

    n, n_slots, rope_rows = (hq + 2 * hkv) * 128, m + 37, 300
    x = randn(m, k + 64).to(dtype)[:, 32:32 + k]
    w = (randn(n, k) * k ** -0.5).to(dtype)
    qn, kn = ((1 + 0.1 * randn(128)).to(dtype) for _ in range(2))
    rope = randn(rope_rows, 128)
    # (positions past the table are clamped, slots that do not exist left out; neither on a 16-byte border)
    pos = torch.randint(-2, rope_rows + 2, (m + 1,), generator=gen, device="cuda")[1:]
    slots = torch.randperm(n_slots, generator=gen, device="cuda")[:m + 1][1:].contiguous()
    slots[m // 2] = -1 if m % 2 else n_slots
    suffix, stream = "_f16" if dtype == torch.float16 else "", ops._stream()
    lib = _lib.load()

    def blank():
        return [torch.full(s, 7.0, dtype=dtype, device="cuda") for s in ((m + 128, hq * 128), (n_slots, hkv, 128), (n_slots, hkv, 128))]

    want, y = blank(), torch.empty((m, n), dtype=dtype, device="cuda")
    _lib.check(getattr(lib, "nvx_internal_prefill_gemm" + suffix)(x.data_ptr(), x.stride(0), w.data_ptr(), y.data_ptr(), m, n, k, 0, 6, stream))
    ops.qknorm_rope_store(y, pos, rope, qn, kn, 1e-6, slots, want[1], want[2], hq, hkv, q_out=want[0][:m])
    assert torch.isfinite(want[0]).all()
    for tile in (10, 5, 14, 15, 0):      # 32, 64, 96 and 128 rows, the rule's
        out = blank()
        _lib.check(getattr(lib, "nvx_internal_prefill_heads" + suffix)(x.data_ptr(), x.stride(0), w.data_ptr(), m, k, tile, pos.data_ptr(), slots.data_ptr(), rope.data_ptr(), rope_rows, n_slots,
                                                                       qn.data_ptr(), kn.data_ptr(), *(o.data_ptr() for o in out), hq, hkv, 1e-6, stream))
        assert all(torch.equal(a, b) for a, b in zip(out, want)), tile
    with pytest.raises(RuntimeError):    # a tile that holds no head
        _lib.check(getattr(lib, "nvx_internal_prefill_heads" + suffix)(x.data_ptr(), x.stride(0), w.data_ptr(), m, k, 6, pos.data_ptr(), slots.data_ptr(), rope.data_ptr(), rope_rows, n_slots,
                                                                       qn.data_ptr(), kn.data_ptr(), *(o.data_ptr() for o in out), hq, hkv, 1e-6, stream))
