// Projections of prefill steps of few hundred tokens: y = x W^T in the 16-bit format, or SiluAndMul of a [gate | up] projection.
//
// Such a product is a few microseconds of matrix work, and what decides its time is how many workgroups the tile leaves to 256 CUs and what a
// workgroup does between two steps of K.  So the tile follows the size, a workgroup keeps STAGES - 1 steps of both operands on their way (memory
// -> LDS without registers, waited for by count, one barrier a step), and the next step's operands are read from LDS while the present one is
// multiplied.  16-byte pieces are XOR-swizzled on the global side.  Small tiles are bound by LDS (a wave reads 3 bytes for every 2 it
// multiplies), which splitting K over the waves would halve; but K is never split: a row's sum runs over K in order, in one chain of
// v_mfma_f32_16x16x32, whatever the tile, so that a token's result does not depend on how many tokens share its step (and equals the library's
// above some 200 rows, whose products take K in the same order).
// The products of a layer of Qwen3-0.6B, us, qkv / o / gate | up / down (the library's without SiluAndMul's own 4 us):
//     64 rows 4.6 / 6.0 / 5.8 / 7.5 (8.8 / 8.4 / 9.0 / 10.1),   216 rows 6.8 / 6.1 / 10.1 / 7.8 (9.4 / 8.9 / 13.4 / 9.4),
//     459 rows 9.1 / 7.9 / 11.8 / 10.0 (11.2 / 9.7 / 13.6 / 12.5),   1536 rows 20.6 / 13.7 / 29.5 / 20.5 (17.7 / 13.7 / 28.9 / 17.1).
#include "prefill_gemm.h"

namespace NVX_NS {

// 64 lanes x 16 bytes from the lanes' addresses to 1 KB of LDS from a wave-uniform address on; the compiler does not count these loads, so every
// wait for them is explicit
__device__ __forceinline__ void piece_to_lds(const void* g, unsigned lds) {
    const unsigned uni = (unsigned)__builtin_amdgcn_readfirstlane((int)lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "s"(uni) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_for_all_but() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }

// TM rows of x by TN rows of w a workgroup of four waves (WM of them along the rows of x), KS columns a step.  With SILU the TN rows of w are 16
// gate and 16 up rows in turn, and the tile gives TN / 2 outputs.  m: rows of x; k % (2 * KS) == 0, n (rows of w) % TN == 0.
template <int TM, int TN, int KS, int STAGES, int WM, bool SILU>
__global__ __launch_bounds__(256) void prefill_gemm_kernel(const uint16_t* __restrict__ x, int64_t x_stride, const uint16_t* __restrict__ w,
                                                          uint16_t* __restrict__ y, int m, int n, int k) {
    constexpr int WN = 4 / WM, FM = TM / WM / 16, FN = TN / WN / 16;       // fragments of a wave
    constexpr int PIECES = KS / 8, AT_ONCE = 64 / PIECES;                  // 16-byte pieces of a row; rows of one copy
    static_assert(PIECES <= 16, "fragments of 16 rows share a swizzle");
    constexpr int ROWS = TM + TN, LOADS = ROWS / AT_ONCE / 4;              // copies of a wave a step
    constexpr int STAGE = ROWS * KS * 2;
    static_assert(ROWS % (4 * AT_ONCE) == 0 && (!SILU || FN % 2 == 0) && (STAGES - 1) * LOADS < 64, "tile");
    constexpr int OUT = SILU ? TN / 2 : TN, LO = OUT + 8;                  // outputs of a row; elements of a row in LDS
    static_assert(TM * LO * 2 <= STAGES * STAGE, "the results turn around in the stages' memory");
    __shared__ __align__(16) unsigned char smem[STAGES * STAGE];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4;
    // tiles are dealt to the XCDs in runs: eight tiles of rows, then the next rows of w
    const int tiles_m = (m + TM - 1) / TM, tiles_n = n / TN, total = tiles_m * tiles_n, per = (total + 7) / 8;
    const int t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || t >= total) return;
    const int group = t / (8 * tiles_n), gm = min(8, tiles_m - group * 8), in = t - group * 8 * tiles_n;
    const int m0 = (group * 8 + in % gm) * TM, tn = in / gm;

    const uint16_t* from[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int r = (wave * LOADS + i) * AT_ONCE + lane / PIECES, c = ((lane % PIECES) ^ (r & (PIECES - 1))) * 8;
        const int rx = min(m0 + r, m - 1), rw = r - TM;                             // (rows past the last repeat it and are not stored)
        const int ww = SILU ? (rw >> 4 & 1) * (n / 2) + tn * OUT + (rw >> 5) * 16 + (rw & 15) : tn * TN + rw;
        from[i] = (r < TM ? x : w) + (int64_t)(r < TM ? rx : ww) * (r < TM ? x_stride : k) + c;
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)smem;
    auto ask = [&](int step) {
        const unsigned at = lds0 + (unsigned)(step % STAGES) * STAGE + wave * LOADS * 1024;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) piece_to_lds(from[i] + (int64_t)step * KS, at + i * 1024);
    };
    const int wm = wave / WN, wn = wave % WN;
    nvx_f32x4 acc[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = nvx_f32x4{0.f, 0.f, 0.f, 0.f};
    typedef __attribute__((address_space(3))) const nvx_u32x4 lds_u4;
    const int steps = k / KS;
    struct Operands { nvx_u32x4 x[KS / 32][FM], w[KS / 32][FN]; };
    auto read = [&](int step, Operands& f) {
        const unsigned base = lds0 + (unsigned)(step % STAGES) * STAGE;
        const unsigned xb = base + (wm * FM * 16 + l16) * (KS * 2), wb = base + (TM + wn * FN * 16 + l16) * (KS * 2);
#pragma unroll
        for (int kk = 0; kk < KS / 32; ++kk) {
            const unsigned off = (unsigned)((4 * kk + quad) ^ (l16 & (PIECES - 1))) * 16;
#pragma unroll
            for (int j = 0; j < FM; ++j) f.x[kk][j] = *reinterpret_cast<lds_u4*>((uintptr_t)(xb + j * 16 * KS * 2 + off));
#pragma unroll
            for (int i = 0; i < FN; ++i) f.w[kk][i] = *reinterpret_cast<lds_u4*>((uintptr_t)(wb + i * 16 * KS * 2 + off));
        }
    };
    // step s is in registers; step s + 1 is read while it is multiplied, and its place in LDS is asked to be filled with step s + STAGES
    auto turn = [&](int s, const Operands& now, Operands& next) {
        if (s + STAGES <= steps) wait_for_all_but<(STAGES - 2) * LOADS>();          // step s + 1 has landed, STAGES - 2 later ones need not have
        else wait_for_all_but<0>();
        __syncthreads();                                                            // everybody's part of it has, and everybody has read step s
        if (s + STAGES < steps) ask(s + STAGES);
        read(s + 1, next);                                                          // (after the last step: whatever lies there, not used)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < KS / 32; ++kk)
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int j = 0; j < FM; ++j) acc[i][j] = mfma_16x16x32_h16(now.w[kk][i], now.x[kk][j], acc[i][j]);
    };
    for (int s = 0; s < STAGES && s < steps; ++s) ask(s);
    if (STAGES <= steps) wait_for_all_but<(STAGES - 1) * LOADS>();
    else wait_for_all_but<0>();
    __syncthreads();
    Operands even, odd;
    read(0, even);
    for (int s = 0; s < steps; s += 2) {
        turn(s, even, odd);
        turn(s + 1, odd, even);
    }
    // a lane has row l16 of every 16 rows of x and four neighbouring outputs (4 * quad ..) of every 16
    __syncthreads();
    uint16_t* so = reinterpret_cast<uint16_t*>(smem);
#pragma unroll
    for (int j = 0; j < FM; ++j) {
        uint16_t* row = so + ((wm * FM + j) * 16 + l16) * LO;
        if constexpr (SILU) {
#pragma unroll
            for (int i = 0; i < FN; i += 2) {
                float o[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = silu_h16(round_h16(acc[i][j][r])) * round_h16(acc[i + 1][j][r]);
                *reinterpret_cast<uint2*>(row + (wn * FN + i) * 8 + 4 * quad) = make_uint2(pack_h16x2(o[0], o[1]), pack_h16x2(o[2], o[3]));
            }
        } else {
#pragma unroll
            for (int i = 0; i < FN; ++i)
                *reinterpret_cast<uint2*>(row + (wn * FN + i) * 16 + 4 * quad) = make_uint2(pack_h16x2(acc[i][j][0], acc[i][j][1]), pack_h16x2(acc[i][j][2], acc[i][j][3]));
        }
    }
    __syncthreads();
    const int cols = SILU ? n / 2 : n;
    for (int p = threadIdx.x; p < TM * OUT / 8; p += 256) {
        const int r = p / (OUT / 8), c = p % (OUT / 8) * 8;
        if (m0 + r < m) *reinterpret_cast<nvx_u32x4*>(y + (int64_t)(m0 + r) * cols + tn * OUT + c) = *reinterpret_cast<const nvx_u32x4*>(so + r * LO + c);
    }
}

template <int TM, int TN, int KS, int STAGES, int WM, bool SILU>
static void launch_prefill_gemm(const void* x, int64_t x_stride, const void* w, void* y, int64_t m, int64_t n, int64_t k, hipStream_t st) {
    const int64_t tiles = (m + TM - 1) / TM * (n / TN);
    hipLaunchKernelGGL((prefill_gemm_kernel<TM, TN, KS, STAGES, WM, SILU>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(256), 0, st, (const uint16_t*)x, x_stride,
                       (const uint16_t*)w, (uint16_t*)y, (int)m, (int)n, (int)k);
}

}  // namespace NVX_NS

using namespace NVX_NS;

static bool nvx_prefill_gemm_fits(int64_t n, int64_t k) { return n > 0 && k > 0 && n % 128 == 0 && k % 256 == 0; }

// The smallest tile whose workgroups all run at once (256 CUs; two a CU for 64 x 64 and for the last) is the fastest at every size measured: us at
// 459 rows of 1024 outputs from 2048 columns, 240 workgroups of 32 x 64: 7.9, 480 of 32 x 32: 8.4, 128 of 64 x 64: 9.9; 300 rows of 4096
// outputs from 1024, 320 of 64 x 64: 8.8, 640 of 32 x 64: 13.6.  Beyond, 64 x 64 in fewer stages (four workgroups a CU) up to 1024 workgroups, then
// 64 x 128 (700 rows of 6144, SiluAndMul: 18.6, 64 x 64 in two stages 23.5).
int NVX_ENTRY(nvx_prefill_gemm)(const void* x, int64_t x_stride, const void* w, void* y, int64_t m, int64_t n, int64_t k, bool silu, hipStream_t st) {
    NVX_REQUIRE(nvx_prefill_gemm_fits(n, k) && m >= 0 && m < (1 << 24) && n < (1 << 24) && k < (1 << 24) && x_stride >= k && x_stride % 8 == 0, NVX_EUNSUPPORTED,
                "nvx_prefill_gemm: sizes");
    NVX_REQUIRE(nvx_aligned16(x) && nvx_aligned16(w) && nvx_aligned16(y), NVX_EINVAL, "nvx_prefill_gemm: pointers must be 16-byte aligned");
    if (m == 0) return NVX_OK;
    auto tiles = [&](int64_t tm, int64_t tn) { return (m + tm - 1) / tm * (n / tn); };
    NVX_REQUIRE(tiles(64, 128) < (1ll << 30), NVX_EUNSUPPORTED, "nvx_prefill_gemm: too many tiles");
    if (silu) {
        if (tiles(32, 64) <= 256) launch_prefill_gemm<32, 64, 128, 4, 2, true>(x, x_stride, w, y, m, n, k, st);
        else if (tiles(64, 64) <= 512) launch_prefill_gemm<64, 64, 64, 4, 2, true>(x, x_stride, w, y, m, n, k, st);
        else if (tiles(64, 64) <= 1024) launch_prefill_gemm<64, 64, 64, 2, 2, true>(x, x_stride, w, y, m, n, k, st);
        else launch_prefill_gemm<64, 128, 64, 2, 2, true>(x, x_stride, w, y, m, n, k, st);
    } else {
        if (tiles(32, 32) <= 256) launch_prefill_gemm<32, 32, 128, 4, 2, false>(x, x_stride, w, y, m, n, k, st);
        else if (tiles(32, 64) <= 256) launch_prefill_gemm<32, 64, 128, 4, 2, false>(x, x_stride, w, y, m, n, k, st);
        else if (tiles(64, 64) <= 512) launch_prefill_gemm<64, 64, 64, 4, 2, false>(x, x_stride, w, y, m, n, k, st);
        else if (tiles(64, 64) <= 1024) launch_prefill_gemm<64, 64, 64, 2, 2, false>(x, x_stride, w, y, m, n, k, st);
        else launch_prefill_gemm<64, 128, 64, 3, 2, false>(x, x_stride, w, y, m, n, k, st);
    }
    return nvx_check_launch("nvx_prefill_gemm");
}
