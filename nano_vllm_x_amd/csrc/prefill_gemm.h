// The products of prefill steps (prefill_gemm.hip, prefill_wide.hip), for the host code that queues them.
#pragma once
#include "rope_dev.h"

// What becomes of a [q | k | v] projection, heads of 128 (hq, hkv and hkv of them): q and k normed per head and turned by their position, q to
// rows of its own (T, hq * 128), k and v to the cache rows `slots` (what nvx_qknorm_rope_store makes of the projection's rows, bit for bit)
struct NvxQkvOut {
    const int64_t *positions, *slots;
    const float* rope;
    int64_t rope_rows, n_slots;
    const uint16_t *q_norm, *k_norm;
    uint16_t *q, *k_cache, *v_cache;
    int hq, hkv;
    float eps;
};
enum { NVX_PG_PLAIN = 0, NVX_PG_SILU = 1, NVX_PG_QKV = 2 };
// tiles; 96_64, 128_64, 160_64, 192_64 and 32_32: not SILU; 32_128 and HEADS_128_128: QKV only; 64_128_THREE (of which a CU has three): SILU only
enum { NVX_PG_256_256 = 1, NVX_PG_192_256, NVX_PG_128_256, NVX_PG_128_128, NVX_PG_64_128, NVX_PG_64_64, NVX_PG_96_64, NVX_PG_32_64, NVX_PG_32_32, NVX_PG_32_128, NVX_PG_128_64, NVX_PG_160_64, NVX_PG_192_64, NVX_PG_96_128, NVX_PG_HEADS_128_128, NVX_PG_160_128, NVX_PG_192_128, NVX_PG_224_128, NVX_PG_64_128_THREE = 20 };

// mode PLAIN: y (m, n) = x (m, k) w (n, k)^T; SILU: y (m, n / 2) = SiluAndMul of it; QKV: the rows of `qkv`, y unused.  In the 16-bit format; rows of x
// `x_stride` elements apart
int NVX_ENTRY(nvx_prefill_gemm)(const void* x, int64_t x_stride, const void* w, void* y, int64_t m, int64_t n, int64_t k, int mode, const NvxQkvOut* qkv,
                                hipStream_t st);
// Whether QKV is the faster way to norm and turn the heads of such a projection, n / 128 of them, than PLAIN and a launch behind it
bool NVX_ENTRY(nvx_prefill_heads_ride)(int64_t m, int64_t n, int64_t k);
// The same, PLAIN or SILU, by the kernel of prefill_wide.hip with tiles of tile_m x tile_n: 256 x 256, 192 x 256, 128 x 256 or 128 x 128; n % tile_n == 0, k % 256 == 0
int NVX_ENTRY(nvx_prefill_wide)(const void* x, int64_t x_stride, const void* w, void* y, int64_t m, int64_t n, int64_t k, bool silu, int tile_m, int tile_n, hipStream_t st);

namespace NVX_NS {

// What a lane of the 16 that hold one head of one token's projection needs of memory for it: asked for before the projection is there
struct QkvHeadIn {
    int64_t slot;
    float4 c, s;
};
__device__ __forceinline__ QkvHeadIn qkv_head_in(int l, int h, int64_t position, int64_t slot, const NvxQkvOut& o) {
    QkvHeadIn in = {h < o.hq ? 0 : slot, {}, {}};
    if (h < o.hq + o.hkv) {
        const float* cs = o.rope + clamp_pos(position, o.rope_rows) * 128 + 4 * l;
        in.c = *reinterpret_cast<const float4*>(cs);
        in.s = *reinterpret_cast<const float4*>(cs + 64);
    }
    return in;
}
// 16 lanes' share of one head of one token's projection: lane l has elements 4 l .. and 64 + 4 l .. as the format holds them, ss the sum of the head's squares,
// wa and wb its norm's weights for them
__device__ __forceinline__ void qkv_head_out(const HalfQuad& x, float ss, const QkvHeadIn& in, const uint2& wa, const uint2& wb, int l, int h, int64_t tok, const NvxQkvOut& o) {
    if (h >= o.hq && (in.slot < 0 || in.slot >= o.n_slots)) return;
    if (h >= o.hq + o.hkv) {
        uint16_t* dst = o.v_cache + (in.slot * o.hkv + (h - o.hq - o.hkv)) * 128 + 4 * l;
        *reinterpret_cast<uint2*>(dst) = make_uint2(pack_h16x2(x.a[0], x.a[1]), pack_h16x2(x.a[2], x.a[3]));
        *reinterpret_cast<uint2*>(dst + 64) = make_uint2(pack_h16x2(x.b[0], x.b[1]), pack_h16x2(x.b[2], x.b[3]));
        return;
    }
    uint16_t* dst = h < o.hq ? o.q + (tok * o.hq + h) * 128 : o.k_cache + (in.slot * o.hkv + (h - o.hq)) * 128;
    *reinterpret_cast<uint4*>(dst + 8 * l) = norm_rotate_interleave(x, ss, wa, wb, o.eps, in.c, in.s);
}
// a lane's part of the sum of squares, as half_quad_sumsq adds it up over 16 lanes
__device__ __forceinline__ float qkv_lane_squares(const HalfQuad& x) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) ss += x.a[j] * x.a[j] + x.b[j] * x.b[j];
    return ss;
}

}  // namespace NVX_NS
