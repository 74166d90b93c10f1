// Products of prefill steps of many tokens: tiles of up to 256 x 256 outputs, with SiluAndMul of a [gate | up] projection at their end.
//
// The walk is wide_dev.h's.  us of 15754 rows, 6144 x 1024 with SiluAndMul 182 (the library's product 159 and silu_mul 50); 4096 x 1024 113 (108),
// 1024 x 2048 54 (49), 1024 x 3072 84 (74);
// of 2160 rows 31 (28 and 9), 22 (29), 17 (19), 24 (24).  Tried and slower: four waves of 128 x 128 (58 where eight are 54), copies in 32-column steps (64).
#include "prefill_gemm.h"
#include "wide_dev.h"

#include <algorithm>

namespace NVX_NS {

struct WideArgs {
    const uint16_t *x, *w;
    uint16_t* y;
    int m, n, k;
    unsigned x_bytes;          // from a row of x to the next
};

// TM rows of x by TN rows of w a tile, STAGES steps on their way.  With SILU a tile's rows of w are 16 gate and 16 up rows in turn (TN / 2 outputs).
// k % 64 == 0 and k / 64 >= STAGES, n (rows of w) % TN == 0.
template <int TM, int TN, int STAGES, int WM, int WN, bool SILU>
__global__ __launch_bounds__(WM * WN * 64) void prefill_wide_kernel(const WideArgs a) {
    typedef WideTile<TM, TN, STAGES, WM, WN> T;
    constexpr int KS = T::KS, FM = T::FM, FN = T::FN, LOADS = T::LOADS, STAGE = T::STAGE, GROUP = 4;   // tiles of rows that share rows of w
    constexpr int OUT = SILU ? TN / 2 : TN, WOUT = OUT / WN, P = WOUT / 8;  // outputs of a row, of a wave's row; 16-byte pieces of that
    constexpr int SIDE = WM * WN * 16 * WOUT * 2;                                      // 16 rows a wave
    static_assert((!SILU || FN % 2 == 0) && (P & (P - 1)) == 0, "tile");
    __shared__ __align__(16) unsigned char smem[STAGES * STAGE + SIDE];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4;
    // the XCDs have runs of tiles: GROUP tiles of rows, then the next rows of w
    const int tiles_m = (a.m + TM - 1) / TM, tiles_n = a.n / TN, total = tiles_m * tiles_n, per = (total + 7) / 8;
    const int last = min(((int)(blockIdx.x & 7) + 1) * per, total), stride = (int)(gridDim.x >> 3);
    int t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (t >= last) return;

    const unsigned w_bytes = 2u * (unsigned)a.k, l8 = lane >> 3, c8 = ((lane & 7) ^ l8) * 16;   // a copy: eight rows, a row's pieces XOR-swizzled
    int m0, tn;
    wide_buffer xb, wb;                    // from the tile's first row of x, of w, to the end (rows of x past the last are zeros, and are not stored)
    auto place = [&]() __attribute__((always_inline)) {
        const int group = t / (GROUP * tiles_n), gm = min(GROUP, tiles_m - group * GROUP), in = t - group * GROUP * tiles_n;
        m0 = (group * GROUP + in % gm) * TM, tn = in / gm;
        xb = wide_buffer_at(reinterpret_cast<const unsigned char*>(a.x) + (int64_t)m0 * a.x_bytes, (int64_t)(a.m - 1 - m0) * a.x_bytes + 2 * a.k);
        wb = wide_buffer_at(reinterpret_cast<const unsigned char*>(a.w) + (int64_t)tn * OUT * w_bytes, 0x7fffffff);
    };
    constexpr bool MIXED = T::MIXED, KEEP = MIXED || LOADS < 8;                                          // offsets of a step's copies stay in registers
    auto of_x = [&](int i) __attribute__((always_inline)) { return (wave * LOADS + (MIXED ? i : 0)) * 8 < TM; };
    auto first_byte = [&](int i) __attribute__((always_inline)) {                      // of a copy, from the tile's first row (scalar)
        const int row = (wave * LOADS + i) * 8, rw = row - TM;
        return of_x(i) ? (unsigned)row * a.x_bytes
                       : (unsigned)(SILU ? (rw >> 4 & 1) * (a.n / 2) + (rw >> 5) * 16 + (rw & 15) : rw) * w_bytes;
    };
    unsigned off[KEEP ? LOADS : 1], from[KEEP ? 1 : LOADS];
    if constexpr (KEEP) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) off[i] = first_byte(i) + l8 * (of_x(i) ? a.x_bytes : w_bytes) + c8;
    } else {
        off[0] = l8 * (of_x(0) ? a.x_bytes : w_bytes) + c8;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) from[i] = (unsigned)__builtin_amdgcn_readfirstlane((int)first_byte(i));
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)smem;
    auto ask = [&](int i, int step, unsigned to) __attribute__((always_inline)) {
        wide_to_lds(of_x(i) ? xb : wb, KEEP ? off[KEEP ? i : 0] : off[0] + from[KEEP ? 0 : i], (unsigned)step * (KS * 2), to);
    };
    const int wm = wave / WN, wn = wave % WN;
    int m_now = 0, tn_now = 0;
    auto finish = [&](nvx_f32x4 (&acc)[FN][FM]) __attribute__((always_inline)) {
        const int r0 = m_now + wm * FM * 16;
        {   // a wave turns 16 rows around at a time, in memory of its own
            unsigned char* so = smem + STAGES * STAGE + wave * 16 * WOUT * 2;
            const int cols = SILU ? a.n / 2 : a.n;
#pragma unroll
            for (int j = 0; j < FM; ++j) {
                auto at = [&](int i) { return reinterpret_cast<uint2*>(so + l16 * (WOUT * 2) + (((2 * i + (quad >> 1)) ^ (l16 & (P - 1))) * 16) + (quad & 1) * 8); };
                if constexpr (SILU) {
#pragma unroll
                    for (int i = 0; i < FN; i += 2) {
                        float o[4];
#pragma unroll
                        for (int r = 0; r < 4; ++r) o[r] = silu_h16(round_h16(acc[i][j][r])) * round_h16(acc[i + 1][j][r]);
                        *at(i / 2) = make_uint2(pack_h16x2(o[0], o[1]), pack_h16x2(o[2], o[3]));
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < FN; ++i) *at(i) = make_uint2(pack_h16x2(acc[i][j][0], acc[i][j][1]), pack_h16x2(acc[i][j][2], acc[i][j][3]));
                }
                wide_lds_wait();
#pragma unroll
                for (int p = 0; p < (16 * P + 63) / 64; ++p) {
                    const int r = (p * 64 + lane) / P, c = lane % P, row = r0 + j * 16 + r;
                    if (r < 16 && row < a.m)
                        *reinterpret_cast<nvx_u32x4*>(a.y + (int64_t)row * cols + tn_now * OUT + wn * WOUT + c * 8) =
                            *reinterpret_cast<const nvx_u32x4*>(so + r * (WOUT * 2) + ((c ^ (r & (P - 1))) * 16));
                }
                wide_lds_wait();
            }
        }
        return t < last;
    };
    place();
    T::walk(lds0, a.k / KS, ask, [&]() __attribute__((always_inline)) { m_now = m0, tn_now = tn; },
            [&]() __attribute__((always_inline)) {
                t += stride;
                if (t < last) place();
            },
            [](nvx_u32x4 w, nvx_u32x4 x, nvx_f32x4 c) __attribute__((always_inline)) { return mfma_16x16x32_h16(w, x, c); }, finish);
}


template <int TM, int TN, int STAGES>
static void launch_prefill_wide(const WideArgs& a, bool silu, hipStream_t st) {
    const int64_t tiles = (int64_t)((a.m + TM - 1) / TM) * (a.n / TN);
    const dim3 grid((unsigned)std::min<int64_t>((tiles + 7) / 8 * 8, 256)), block(512);        // (a workgroup a CU: its LDS)
    if (silu) hipLaunchKernelGGL((prefill_wide_kernel<TM, TN, STAGES, 2, 4, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((prefill_wide_kernel<TM, TN, STAGES, 2, 4, false>), grid, block, 0, st, a);
}

}  // namespace NVX_NS

using namespace NVX_NS;

int NVX_ENTRY(nvx_prefill_wide)(const void* x, int64_t x_stride, const void* w, void* y, int64_t m, int64_t n, int64_t k, bool silu, int tile_m, int tile_n, hipStream_t st) {
    // a buffer's bytes and offsets are 31 bits wide: TM rows of x, the rows of w
    NVX_REQUIRE(m > 0 && m < (1 << 24) && n > 0 && tile_n > 0 && n % tile_n == 0 && k >= 256 && k % 256 == 0 && x_stride >= k && x_stride < (1 << 21) && n * k < (1ll << 30) &&
                (m + 127) / 128 * (n / 128) < (1ll << 30), NVX_EUNSUPPORTED, "nvx_prefill_wide: sizes");
    const WideArgs a = {(const uint16_t*)x, (const uint16_t*)w, (uint16_t*)y, (int)m, (int)n, (int)k, (unsigned)(2 * x_stride)};
    if (tile_m == 256 && tile_n == 256) launch_prefill_wide<256, 256, 2>(a, silu, st);
    else if (tile_m == 192 && tile_n == 256) launch_prefill_wide<192, 256, 2>(a, silu, st);
    else if (tile_m == 128 && tile_n == 256) launch_prefill_wide<128, 256, 2>(a, silu, st);
    else if (tile_m == 128 && tile_n == 128) launch_prefill_wide<128, 128, 4>(a, silu, st);
    else return nvx_fail(NVX_EUNSUPPORTED, "nvx_prefill_wide: no tile of %d x %d", tile_m, tile_n);
    return nvx_check_launch("nvx_prefill_wide");
}
