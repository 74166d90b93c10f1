// Products of prefill steps of many tokens: tiles of up to 256 x 256 outputs, with SiluAndMul of a [gate | up] projection at their end.
//
// Such a product is bound by its matrix instructions (65 % of the kernel's clocks in each, at 2.0 GHz or less under full load) and, next to them, by LDS, of which
// eight waves read 1.5 bytes for every 512 operations.  So everything is dealt out evenly: a step is 64 columns of K, both operands memory -> LDS without
// registers, two or four steps on their way; in each half of a step a wave multiplies 32 columns while it reads the next 32, and one barrier a step, between the halves, says that a
// step has landed everywhere and that its predecessor may be overwritten.  Copies are asked for one between every four products: all at once they stop the
// wave that asks (15754 x 1024 x 2048: 56.2 us, dealt out 53.3); their addresses are a buffer's, so that a copy costs two scalar instructions and at most one of the
// vector's, and rows past the last read zeros.  A workgroup takes its share of the tiles without a pause: the last steps of a tile ask for the first of the next, and
// results turn around in LDS of their own.  K is in order, one chain of v_mfma_f32_16x16x32 an output, as in prefill_gemm.hip.
// us of 15754 rows, 6144 x 1024 with SiluAndMul 182 (the library's product 159 and silu_mul 50); 4096 x 1024 113 (108), 1024 x 2048 54 (49), 1024 x 3072 84 (74);
// of 2160 rows 31 (28 and 9), 22 (29), 17 (19), 24 (24).  Tried and slower: four waves of 128 x 128 (58 where eight are 54), copies in 32-column steps (64).
#include "prefill_gemm.h"

#include <algorithm>
#include <type_traits>

namespace NVX_NS {

// 64 lanes x 16 bytes from the lanes' byte offsets (and `step`) into a buffer to 1 KB of LDS from `lds` on, both wave-uniform; lanes past the buffer's end
// read zeros.  The compiler does not count these loads, so every wait for them is explicit
typedef int wide_buffer __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void wide_to_lds(wide_buffer buf, unsigned off, unsigned step, unsigned lds) {
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" : : "v"(off), "s"(buf), "s"(step), "s"(lds) : "memory");
}
__device__ __forceinline__ wide_buffer wide_buffer_at(const void* base, int64_t bytes) {
    const uint64_t at = (uint64_t)base;
    return wide_buffer{(int)(uint32_t)at, (int)(uint32_t)(at >> 32), (int)(uint32_t)(bytes < 0x7fffffffll ? bytes : 0x7fffffffll), 0x00020000};
}
template <int N>
__device__ __forceinline__ void wide_wait_for_all_but() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }
__device__ __forceinline__ void wide_lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory"); }

struct WideArgs {
    const uint16_t *x, *w;
    uint16_t* y;
    int m, n, k;
    unsigned x_bytes;          // from a row of x to the next
};

// TM rows of x by TN rows of w a tile, STAGES steps on their way, WM x WN waves.  With SILU a tile's rows of w are 16 gate and 16 up rows in turn (TN / 2 outputs).
// k % 64 == 0 and k / 64 >= STAGES, n (rows of w) % TN == 0.
template <int TM, int TN, int STAGES, int WM, int WN, bool SILU>
__global__ __launch_bounds__(WM * WN * 64) void prefill_wide_kernel(const WideArgs a) {
    constexpr int KS = 64, FM = TM / WM / 16, FN = TN / WN / 16, EACH = 4, GROUP = 4;   // fragments of a wave; products between two copies; tiles of rows that share rows of w
    constexpr int LOADS = (TM + TN) / 8 / (WM * WN), STAGE = (TM + TN) * KS * 2;                  // copies of a wave a step
    constexpr int OUT = SILU ? TN / 2 : TN, WOUT = OUT / WN, P = WOUT / 8;  // outputs of a row, of a wave's row; 16-byte pieces of that
    constexpr int SIDE = WM * WN * 16 * WOUT * 2;                                      // 16 rows a wave
    static_assert((TM + TN) % (8 * WM * WN) == 0 && FM * FN % EACH == 0 && (!SILU || FN % 2 == 0) && (P & (P - 1)) == 0, "tile");
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
    constexpr bool MIXED = TM / 8 % LOADS != 0;                                        // a wave copies rows of both
    constexpr bool KEEP = MIXED || LOADS < 8;                                          // offsets of a step's copies stay in registers
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
    auto ask = [&](int i, int step, int slot) __attribute__((always_inline)) {
        wide_to_lds(of_x(i) ? xb : wb, KEEP ? off[KEEP ? i : 0] : off[0] + from[KEEP ? 0 : i], (unsigned)step * (KS * 2),
                    lds0 + (unsigned)slot * STAGE + (wave * LOADS + i) * 1024);
    };
    const int wm = wave / WN, wn = wave % WN;
    nvx_f32x4 acc[FN][FM];
    typedef __attribute__((address_space(3))) const nvx_u32x4 lds_u4;
    const int steps = a.k / KS;
    struct Operands { nvx_u32x4 x[FM], w[FN]; };
    const unsigned xl = lds0 + (wm * FM * 16 + l16) * (KS * 2), wl = lds0 + (TM + wn * FN * 16 + l16) * (KS * 2);
    const unsigned piece[2] = {(unsigned)(quad ^ (l16 & 7)) * 16, (unsigned)((4 + quad) ^ (l16 & 7)) * 16};
    auto read = [&](int q, unsigned off, Operands& f) __attribute__((always_inline)) {
        if (q < FM) f.x[q] = *reinterpret_cast<lds_u4*>((uintptr_t)(xl + off + q * 16 * KS * 2));
        else f.w[q - FM] = *reinterpret_cast<lds_u4*>((uintptr_t)(wl + off + (q - FM) * 16 * KS * 2));
    };
    // half a step: `now` is multiplied, `next` read (the half of the step in `slot` that FIRST says), with FIRST the step `asked` asked for
    auto half = [&](const Operands& now, Operands& next, int slot, auto first, int asked, int ask_slot) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first)::value;
        constexpr int READS = FM + FN, CHUNKS = FM * FN / EACH, R = CHUNKS >= 8 ? CHUNKS - 2 : CHUNKS;     // (the reads end before the products do)
        const unsigned off = piece[FIRST ? 0 : 1] + (unsigned)slot * STAGE;
#pragma unroll
        for (int i = 0; i < CHUNKS; ++i) {
#pragma unroll
            for (int q = 0; q < READS; ++q)
                if (q * R / READS == i) read(q, off, next);
            if constexpr (FIRST) {
#pragma unroll
                for (int q = 0; q < LOADS; ++q)
                    if (q * CHUNKS / LOADS == i) ask(q, asked, ask_slot);
            }
#pragma unroll
            for (int u = i * EACH; u < (i + 1) * EACH; ++u) acc[u / FM][u % FM] = mfma_16x16x32_h16(now.w[u / FM], now.x[u % FM], acc[u / FM][u % FM]);
            __builtin_amdgcn_sched_barrier(0);
        }
        wide_lds_wait();
        __builtin_amdgcn_sched_barrier(0);
    };
    place();
    for (int s = 0; s < STAGES; ++s)
#pragma unroll
        for (int i = 0; i < LOADS; ++i) ask(i, s, s);
    Operands even, odd;
    int slot = 0;
    wide_wait_for_all_but<(STAGES - 1) * LOADS>();
    __syncthreads();
#pragma unroll
    for (int q = 0; q < FM + FN; ++q) read(q, piece[0], even);
    wide_lds_wait();
    for (;;) {
        const int m_now = m0, tn_now = tn;
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int j = 0; j < FM; ++j) acc[i][j] = nvx_f32x4{0.f, 0.f, 0.f, 0.f};
        int asked = STAGES;
        for (int s = 0; s < steps; ++s) {
            half(even, odd, slot, std::false_type{}, 0, 0);
            wide_wait_for_all_but<(STAGES - 2) * LOADS>();          // the step behind this one has landed (stores of a tile before count too, and are older)
            __builtin_amdgcn_s_barrier();                           // everybody's part of it has, and everybody has read this one (wide_lds_wait)
            asm volatile("" : : : "memory");
            const int was = slot;
            slot = slot + 1 == STAGES ? 0 : slot + 1;
            if (asked == steps) {                                   // the next tile's first steps (behind the last tile: this one's again, not used)
                asked = 0, t += stride;
                if (t < last) place();
            }
            half(odd, even, slot, std::true_type{}, asked, was);
            ++asked;
        }
        // a lane has row l16 of every 16 rows of x and four neighbouring outputs (4 * quad ..) of every 16
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
        if (t >= last) break;
    }
    wide_wait_for_all_but<0>();      // (nothing may still be on its way to this memory when it is another workgroup's)
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
