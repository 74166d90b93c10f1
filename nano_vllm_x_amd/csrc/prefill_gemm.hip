// Projections of prefill steps: y = x W^T in the 16-bit format, SiluAndMul of a [gate | up] projection, or what becomes of a [q | k | v] projection
// (NvxQkvOut); here the kernel for few hundred tokens and the choice between it and those for many (prefill_wide.hip).
//
// Such a product is a few microseconds of matrix work, and what decides its time is how many workgroups the tile leaves to 256 CUs and what a
// workgroup does between two steps of K.  So the tile follows the size, a workgroup keeps STAGES - 1 steps of both operands on their way (memory
// -> LDS without registers, waited for by count, one barrier a step), and the next step's operands are read from LDS while the present one is
// multiplied.  16-byte pieces are XOR-swizzled on the global side.  Small tiles are bound by what they bring into a CU (see PREFILL_TILES) and by LDS (a wave reads 3 bytes for every 2
// it multiplies), which splitting K over the waves would halve; but K is never split: a row's sum runs over K in order, in one chain of
// v_mfma_f32_16x16x32, whatever the tile, so that a token's result does not depend on how many tokens share its step (and equals the library's
// above some 200 rows, whose products take K in the same order).
// The products of a layer of Qwen3-0.6B with weights that no cache holds, one kind of product behind another of its kind, us, qkv / o / gate | up / down: 100 rows 5.6 / 6.2 / 7.4 / 8.2, 200 rows 7.0 / 6.3 / 9.5 / 8.3,
//     459 rows 9.1 / 8.2 / 12.1 / 11.2, 1500 rows 18.0 / 12.6 / 29.2 / 18.0 (by the same measure before copies and reads were dealt out and there were tiles of 96 to 224 x 128: 100 rows 5.9 / 6.5 / 7.6 / 8.4, 200 7.2 / 6.6 / 10.5 /
//     8.5, 459 10.6 / 8.5 / 12.9 / 11.4, 1500 24.0 / 13.0 / 29.2 / 18.3; the library with weights in its caches: 64 rows 8.8 / 8.4 / 9.0 and SiluAndMul's 4 / 10.1, 459 rows
//     11.2 / 9.7 / 13.6 and 4 / 12.5, 1536 rows 17.7 / 13.7 / 28.9 and 4 / 17.1).  Within a step 459 rows take 12.5 with the heads' norms and rotations, 13.4 for gate | up, 9.95 in the mean of o and down.
#include "prefill_gemm.h"

#include <type_traits>

namespace NVX_NS {

// 64 lanes x 16 bytes from the lanes' addresses to 1 KB of LDS from a wave-uniform address on; the compiler does not count these loads, so every
// wait for them is explicit
__device__ __forceinline__ void piece_to_lds(const void* g, unsigned lds) {
    const unsigned uni = (unsigned)__builtin_amdgcn_readfirstlane((int)lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "s"(uni) : "memory");
}
// 64 lanes x 4 bytes likewise
__device__ __forceinline__ void words_to_lds(const void* g, unsigned lds) {
    const unsigned uni = (unsigned)__builtin_amdgcn_readfirstlane((int)lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(g), "s"(uni) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_for_all_but() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }

// TM rows of x by TN rows of w a workgroup of four waves (WM of them along the rows of x), KS columns a step.  With SILU the TN rows of w are 16
// gate and 16 up rows in turn, and the tile gives TN / 2 outputs; with QKV a tile is one head.  m: rows of x; k % (2 * KS) == 0, n (rows of w) % TN == 0.
template <int TM, int TN, int KS, int STAGES, int WM, int MODE>
__global__ __launch_bounds__(256, STAGES == 2 ? 3 : 1) void prefill_gemm_kernel(const uint16_t* __restrict__ x, int64_t x_stride, const uint16_t* __restrict__ w,
                                                          uint16_t* __restrict__ y, int m, int n, int k, const NvxQkvOut qkv) {
    constexpr bool SILU = MODE == NVX_PG_SILU;
    constexpr int WN = 4 / WM, FM = TM / WM / 16, FN = TN / WN / 16;       // fragments of a wave
    constexpr int PIECES = KS / 8, AT_ONCE = 64 / PIECES;                  // 16-byte pieces of a row; rows of one copy
    static_assert(PIECES <= 16, "fragments of 16 rows share a swizzle");
    constexpr int ROWS = TM + TN, LOADS = ROWS / AT_ONCE / 4;              // copies of a wave a step
    constexpr int STAGE = ROWS * KS * 2;
    static_assert(STAGES >= 2 && STAGES <= 4, "the last steps are written out");
    static_assert(ROWS % (4 * AT_ONCE) == 0 && (!SILU || FN % 2 == 0) && (MODE != NVX_PG_QKV || TN == 128) && (STAGES - 1) * LOADS < 64, "tile");
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
    // one of a wave's copies of a step, then its next step's place
    auto ask = [&](int i, unsigned slot) __attribute__((always_inline)) {
        piece_to_lds(from[i], lds0 + slot + (wave * LOADS + i) * 1024);
        from[i] += KS;
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
    constexpr int EACH = FM + FN, READS = KS / 32 * EACH, MULS = KS / 32 * FM * FN, EARLY = MULS >= 8 ? MULS * 5 / 8 : MULS;   // the reads are among the first EARLY products
    const unsigned xl = lds0 + (wm * FM * 16 + l16) * (KS * 2), wl = lds0 + (TM + wn * FN * 16 + l16) * (KS * 2);
    auto read = [&](int q, unsigned slot, Operands& f) __attribute__((always_inline)) {
        const int kk = q / EACH, i = q % EACH;
        const unsigned off = slot + (unsigned)((4 * kk + quad) ^ (l16 & (PIECES - 1))) * 16;
        if (i < FM) f.x[kk][i] = *reinterpret_cast<lds_u4*>((uintptr_t)(xl + i * 16 * KS * 2 + off));
        else f.w[kk][i - FM] = *reinterpret_cast<lds_u4*>((uintptr_t)(wl + (i - FM) * 16 * KS * 2 + off));
    };
    unsigned slot = 0;                                                              // of step s
    // Step s is in registers; step s + 1 is read while it is multiplied, and its place in LDS is asked to be filled with step s + STAGES (ASKS).  Copies and reads are dealt
    // out between the products: a wave that asks for all its copies at once waits for as long as the CU takes them in (64 bytes a clock), and multiplies nothing meanwhile.
    // FLYING: copies of later steps than s + 1 that need not have landed; LAST: there is no step s + 1.
    auto turn = [&](auto flying, auto asks, auto last, const Operands& now, Operands& next) __attribute__((always_inline)) {
        constexpr bool ASKS = decltype(asks)::value, LAST = decltype(last)::value;
        const unsigned free_slot = slot;
        slot = slot == (STAGES - 1) * STAGE ? 0 : slot + STAGE;
        if (!LAST) {
            wait_for_all_but<decltype(flying)::value>();                            // step s + 1 has landed
            asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");                    // and this wave has read step s (a barrier alone does not wait for reads)
            __syncthreads();                                                        // everybody's part of it has, and everybody has read step s
        }
#pragma unroll
        for (int u = 0; u < MULS; ++u) {
            const int kk = u / (FM * FN), i = u / FM % FN, j = u % FM;
            if (!LAST) {
#pragma unroll
                for (int q = 0; q < READS; ++q)
                    if (q * EARLY / READS == u) read(q, slot, next);
            }
            if (ASKS) {
#pragma unroll
                for (int q = 0; q < LOADS; ++q)
                    if (q * MULS / LOADS == u) ask(q, free_slot);
            }
            acc[i][j] = mfma_16x16x32_h16(now.w[kk][i], now.x[kk][j], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // QKV: where the tile's tokens stand and what their heads' ends read of memory.  Positions and slots come ahead of all copies, into LDS (a wave's wait for a step
    // covers its older copies); what they lead to is on its way during the last steps.  459 tokens of Qwen3-0.6B, us a step: 1979 with tiles of 32 rows, two a CU, whose ends read one after
    // the other; 1903 with one of 64.
    constexpr bool HEADS = MODE == NVX_PG_QKV;
    __shared__ int64_t where[HEADS ? 2 * TM : 1];
    QkvHeadIn foreseen[HEADS ? TM / 16 : 1];
    uint2 wa = {}, wb = {};
    if constexpr (HEADS) {
        static_assert(TM % 32 == 0, "a copy is 32 tokens");
        for (int c = wave; c < TM / 16; c += 4) {
            const bool first = c < TM / 32;
            words_to_lds(reinterpret_cast<const int32_t*>(first ? qkv.positions : qkv.slots) + 2 * min(m0 + (first ? c : c - TM / 32) * 32 + (lane >> 1), m - 1) + (lane & 1),
                         (unsigned)(uintptr_t)(const __attribute__((address_space(3))) int64_t*)where + c * 256);
        }
    }
    auto foresee = [&]() __attribute__((always_inline)) {
        if constexpr (HEADS) {
            const uint16_t* const norm = tn < qkv.hq ? qkv.q_norm : qkv.k_norm;
            wa = *reinterpret_cast<const uint2*>(norm + 4 * l16);
            wb = *reinterpret_cast<const uint2*>(norm + 64 + 4 * l16);
#pragma unroll
            for (int i = 0; i < TM / 16; ++i) {
                const int r = (int)(threadIdx.x >> 4) + 16 * i;
                foreseen[i] = qkv_head_in(l16, tn, where[r], where[TM + r], qkv);
            }
        }
    };
    const int begun = min(STAGES, steps);
    for (int s = 0; s < begun; ++s)
#pragma unroll
        for (int i = 0; i < LOADS; ++i) ask(i, s * STAGE);
    std::true_type yes;
    std::false_type no;
    Operands even, odd;
    if (STAGES <= steps) wait_for_all_but<(STAGES - 1) * LOADS>();
    else wait_for_all_but<0>();
    __syncthreads();
#pragma unroll
    for (int q = 0; q < READS; ++q) read(q, 0, even);
    if constexpr (STAGES == 2) {
        // Three workgroups a CU, of which each multiplies while the others wait: all copies and reads of a step at once.  Dealt out they take 204 registers, and a SIMD with three waves has 168 for each.
        auto plain_turn = [&](int s, const Operands& now, Operands& next) __attribute__((always_inline)) {
            wait_for_all_but<0>();
            asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
            __syncthreads();                                                        // step s + 1 has landed, and everybody has read step s
            if (s + 2 < steps) {
#pragma unroll
                for (int i = 0; i < LOADS; ++i) ask(i, slot);
            }
            slot ^= STAGE;
#pragma unroll
            for (int q = 0; q < READS; ++q) read(q, slot, next);                    // (behind the last step whatever lies there: not used)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < MULS; ++u) {
                const int kk = u / (FM * FN), i = u / FM % FN, j = u % FM;
                acc[i][j] = mfma_16x16x32_h16(now.w[kk][i], now.x[kk][j], acc[i][j]);
            }
        };
        for (int s = 0; s < steps; s += 2) {                                        // (k / KS is even)
            plain_turn(s, even, odd);
            plain_turn(s + 1, odd, even);
        }
    } else if (steps < STAGES) {                                                    // (k / KS is even)
        foresee();
        std::integral_constant<int, 0> none;
        for (int s = 0; s + 2 < steps; s += 2) {
            turn(none, no, no, even, odd);
            turn(none, no, no, odd, even);
        }
        turn(none, no, no, even, odd);
        turn(none, no, yes, odd, even);
    } else {
        std::integral_constant<int, (STAGES - 2) * LOADS> most;
        int left = steps - STAGES;
        for (; left > 1; left -= 2) {
            turn(most, yes, no, even, odd);
            turn(most, yes, no, odd, even);
        }
        auto rest = [&](Operands& now, Operands& next) __attribute__((always_inline)) {     // the last STAGES steps, which have all been asked for
            auto one = [&](auto j, Operands& a, Operands& b) __attribute__((always_inline)) {
                constexpr int J = decltype(j)::value, F = STAGES - 2 - J;
                if constexpr (J < STAGES) turn(std::integral_constant<int, (F > 0 ? F : 0) * LOADS>{}, no, std::integral_constant<bool, J == STAGES - 1>{}, a, b);
            };
            one(std::integral_constant<int, 0>{}, now, next);
            one(std::integral_constant<int, 1>{}, next, now);
            one(std::integral_constant<int, 2>{}, now, next);
            one(std::integral_constant<int, 3>{}, next, now);
        };
        if constexpr (STAGES % 2) {
            turn(most, yes, no, even, odd);
            foresee();
            rest(odd, even);
        } else {
            foresee();
            rest(even, odd);
        }
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
    if constexpr (MODE == NVX_PG_QKV) {
#pragma unroll
        for (int i = 0; i < TM / 16; ++i) {
            const int r = (int)(threadIdx.x >> 4) + 16 * i;
            const HalfQuad hq = load_half_quads(so + r * LO, l16);
            const float ss = quarter_sum(qkv_lane_squares(hq));
            if (m0 + r < m) qkv_head_out(hq, ss, foreseen[i], wa, wb, l16, tn, m0 + r, qkv);
        }
        return;
    }
    const int cols = SILU ? n / 2 : n;
    for (int p = threadIdx.x; p < TM * OUT / 8; p += 256) {
        const int r = p / (OUT / 8), c = p % (OUT / 8) * 8;
        if (m0 + r < m) *reinterpret_cast<nvx_u32x4*>(y + (int64_t)(m0 + r) * cols + tn * OUT + c) = *reinterpret_cast<const nvx_u32x4*>(so + r * LO + c);
    }
}

template <int TM, int TN, int KS, int STAGES, int WM, int MODE>
static void launch_prefill_gemm(const void* x, int64_t x_stride, const void* w, void* y, int64_t m, int64_t n, int64_t k, const NvxQkvOut* qkv, hipStream_t st) {
    const int64_t tiles = (m + TM - 1) / TM * (n / TN);
    hipLaunchKernelGGL((prefill_gemm_kernel<TM, TN, KS, STAGES, WM, MODE>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(256), 0, st, (const uint16_t*)x, x_stride,
                       (const uint16_t*)w, (uint16_t*)y, (int)m, (int)n, (int)k, MODE == NVX_PG_QKV ? *qkv : NvxQkvOut{});
}

}  // namespace NVX_NS

using namespace NVX_NS;

// What a tile costs, us, with weights that no cache holds: us + (rounds - 1) * again + k / 1024 * (us_k + (rounds - 1) * round + (workgroups / 256 - 1) * over), rounds of 256 workgroups and the last
// term from the 257th on (us_k 0: not built).  Plain: fitted to 40 to 4000 rows of 1024 to 12288 outputs of 512 to 3072 columns, with `again` 0; of 813 products of 30 to 8000 rows of 256 to 8192 columns
// the tile it picks costs 0.7 % more than the best one (the tiles and costs before 7 %).  SiluAndMul: fitted to 1 365 products of 30 to 18 000 rows, 256 to 2048 columns; over 1 358 others its choice is 0.2 % off the best (15 % at worst); without `again`, what
// a round costs however few its columns are (results, SiluAndMul, first copies), narrow layers got tiles 5 to 45 % off.  A step of a few KB is as long as its copies' way into a CU, its reads from LDS and two barriers'
// skew, hardly any of which hides any other at one workgroup a CU, so the tile that just fills the CUs is the best, and there is one for most sizes: without the tiles of 96 to 224 x 128, and with
// two and three steps of 64 x 128 in LDS, the choice was 6 % and 8 % off.  us a product without and with them: SiluAndMul's 6144 x 1024, 256 rows 11.7 and 10.4 (64 x 128), 768 20.2 and 16.5 (160 x 128), 900 20.7 and 18.3, 1024 21.9 and 19.2;
// 4096 x 1024, 1200 rows 23.0 and 15.7, 1500 23.9 and 17.6; 2048 x 2048, 3072 rows 42.7 and 27.9; 12288 x 2048, 300 rows 35.6 and 26.9.  256 x 128 needs more registers than there are.  A deeper
// ring (all of LDS) was no faster; nor were rows of w a multiple of 128 bytes and 64 apart.
// 64_128_THREE: three workgroups a CU, where all of them run at once (768; `again` and `round` for every 256 past the first), which is the best for narrow layers: SiluAndMul's 1536 x 256, 4096 rows 8.1 and by the best
// of the others 9.6; 3072 x 256, 1836 rows 8.0 and 9.0; 3072 x 512, 2048 rows 12.3 and 12.9; 1024 x 512, 5300 rows 11.0 and 11.5.
struct PrefillCost { float us, again, us_k, round, over; };
struct PrefillTile { int tile, m, n; PrefillCost plain, silu; bool wide; };
static const PrefillTile PREFILL_TILES[] = {
    {NVX_PG_32_32, 32, 32, {2.1f, 0.f, 2.05f, 1.2f, .4f}, {}, false},
    {NVX_PG_32_64, 32, 64, {2.3f, 0.f, 2.9f, 2.35f, 1.1f}, {2.49f, 1.4f, 3.51f, 3.3f, -.15f}, false},
    {NVX_PG_64_64, 64, 64, {2.2f, 0.f, 4.2f, 2.f, 1.45f}, {2.07f, .51f, 5.51f, 1.97f, 1.01f}, false},
    {NVX_PG_96_64, 96, 64, {2.7f, 0.f, 4.7f, 2.8f, 1.75f}, {}, false},
    {NVX_PG_128_64, 128, 64, {3.1f, 0.f, 5.2f, 5.5f, 1.5f}, {}, false},
    {NVX_PG_160_64, 160, 64, {3.5f, 0.f, 6.1f, 6.f, 2.6f}, {}, false},
    {NVX_PG_192_64, 192, 64, {3.8f, 0.f, 7.f, 7.1f, 2.4f}, {}, false},
    {NVX_PG_64_128, 64, 128, {2.8f, 0.f, 6.f, 5.55f, 1.3f}, {3.06f, 2.24f, 7.24f, 5.09f, .26f}, false},
    {NVX_PG_64_128_THREE, 64, 128, {}, {2.33f, .88f, 13.23f, 1.54f, 0.f}, false},
    {NVX_PG_96_128, 96, 128, {3.6f, 0.f, 7.25f, 6.6f, 2.3f}, {3.82f, 3.12f, 7.55f, 5.31f, 1.09f}, false},
    {NVX_PG_128_128, 128, 128, {4.f, 0.f, 7.7f, 6.65f, 2.3f}, {4.37f, 2.08f, 8.85f, 6.12f, 1.54f}, true},
    {NVX_PG_160_128, 160, 128, {5.f, 0.f, 9.4f, 10.3f, 1.9f}, {5.52f, 4.14f, 10.18f, 8.66f, 1.27f}, false},
    {NVX_PG_192_128, 192, 128, {5.3f, 0.f, 10.9f, 10.75f, 3.3f}, {6.08f, 4.79f, 10.69f, 8.47f, 2.44f}, false},
    {NVX_PG_224_128, 224, 128, {5.35f, 0.f, 11.9f, 11.15f, 6.8f}, {6.48f, 5.05f, 12.48f, 9.56f, 2.79f}, false},
    {NVX_PG_128_256, 128, 256, {.7f, 0.f, 21.4f, 13.6f, 3.7f}, {4.41f, 3.44f, 21.14f, 10.54f, 3.89f}, true},
    {NVX_PG_192_256, 192, 256, {1.7f, 0.f, 23.2f, 14.3f, 8.6f}, {6.68f, 5.94f, 22.64f, 10.51f, 6.78f}, true},
    {NVX_PG_256_256, 256, 256, {4.9f, 0.f, 23.8f, 12.f, 10.f}, {8.95f, 7.72f, 23.45f, 12.06f, 9.64f}, true}};

// QKV, a tile as wide as a head, in one round of workgroups: us + k / 1024 * us_k, less what the launch costs that norms and turns the heads behind a plain product (the two grow alike with
// the rows).  Fitted to steps of 20 to 1024 tokens of layers of 512 to 2560: these costs, held against the plain tiles', were right wherever the two ways differ by more than
// 1 us a layer.  us a layer of 1024 columns and 32 heads, plain and launch / here: 130 tokens 55.9 / 54.5, 256 61.3 / 59.8 (32 rows), 300 66.1 / 65.2, 459 73.4 / 71.3 (64 rows), 768 98.2 / 94.0 (96), 900
// 98.5 / 96.8 (128), 64 49.6 / 50.8, not taken; 2048 columns: 300 115.0 / 116.2, not taken, 400 117.3 / 116.0.  In two rounds the plain tiles lead (96 rows at 1500 tokens by some 1 us).
// Two workgroups a CU were never the better way, nor steps of 128 columns.  A 256 x 256 tile's heads take 15 us, in which its CU multiplies nothing.
struct HeadsTile { int tile, m; float us, us_k; };
static const HeadsTile HEADS_TILES[] = {{NVX_PG_32_128, 32, -.4f, 5.3f}, {NVX_PG_64_128, 64, .1f, 6.3f}, {NVX_PG_96_128, 96, .9f, 6.4f}, {NVX_PG_HEADS_128_128, 128, 2.4f, 7.7f}};
static int heads_tile(int64_t m, int64_t n, int64_t k, float& cost) {
    int best = 0;
    for (const HeadsTile& t : HEADS_TILES) {
        if ((m + t.m - 1) / t.m * (n / 128) > 256) continue;
        const float c = t.us + (float)k / 1024.f * t.us_k;
        if (!best || c < cost) best = t.tile, cost = c;
    }
    return best;
}

// The least of the first table's.
static int prefill_gemm_rule(int64_t m, int64_t n, int64_t k, bool silu, bool wide, float& least) {
    int best = NVX_PG_64_64;
    least = 0.f;
    for (const PrefillTile& t : PREFILL_TILES) {
        const PrefillCost& c = silu ? t.silu : t.plain;
        if (c.us_k == 0.f || n % t.n || (t.wide && !wide)) continue;
        const int64_t workgroups = (m + t.m - 1) / t.m * (n / t.n);
        if (t.tile == NVX_PG_64_128_THREE && workgroups > 768) continue;
        const float past = workgroups > 256 ? (float)workgroups / 256.f - 1.f : 0.f, rounds = t.tile == NVX_PG_64_128_THREE ? past : (float)((workgroups + 255) / 256 - 1);      // past the first
        const float cost = c.us + rounds * c.again + (float)k / 1024.f * (c.us_k + rounds * c.round + past * c.over);
        if (least == 0.f || cost < least) best = t.tile, least = cost;
    }
    return best;
}

bool NVX_ENTRY(nvx_prefill_heads_ride)(int64_t m, int64_t n, int64_t k) {
    float here = 0.f, plain;
    if (!heads_tile(m, n, k, here)) return false;
    prefill_gemm_rule(m, n, k, false, n * k < (1ll << 30), plain);
    return here < plain;
}

// tile: one of NVX_PG_*, or 0 by the rule
static int prefill_gemm(int tile, const void* x, int64_t x_stride, const void* w, void* y, int64_t m, int64_t n, int64_t k, int mode, const NvxQkvOut* qkv, hipStream_t st) {
    NVX_REQUIRE(mode >= NVX_PG_PLAIN && mode <= NVX_PG_QKV && n > 0 && k > 0 && n % 128 == 0 && k % 256 == 0 && m >= 0 && m < (1 << 24) && n < (1 << 24) && k < (1 << 24) &&
                x_stride >= k && x_stride % 8 == 0, NVX_EUNSUPPORTED, "nvx_prefill_gemm: sizes");
    NVX_REQUIRE(mode != NVX_PG_QKV || (qkv && n == (int64_t)(qkv->hq + 2 * qkv->hkv) * 128), NVX_EINVAL, "nvx_prefill_gemm: heads");
    NVX_REQUIRE(x && w && (y || mode == NVX_PG_QKV) && nvx_aligned16(x) && nvx_aligned16(w) && nvx_aligned16(y), NVX_EINVAL, "nvx_prefill_gemm: pointers must be 16-byte aligned");
    if (m == 0) return NVX_OK;
    NVX_REQUIRE((m + 31) / 32 * (n / 32) < (1ll << 30), NVX_EUNSUPPORTED, "nvx_prefill_gemm: too many tiles");
    const bool silu = mode == NVX_PG_SILU;
    float cost;
    if (tile == 0 && mode == NVX_PG_QKV) {
        tile = heads_tile(m, n, k, cost);
        if (!tile) tile = NVX_PG_32_128;
    } else if (tile == 0) tile = prefill_gemm_rule(m, n, k, silu, x_stride < (1 << 21) && n * k < (1ll << 30), cost);       // (what the wide tiles' offsets hold)
    if (mode != NVX_PG_QKV && tile >= NVX_PG_256_256 && tile < NVX_PG_64_128)
        return NVX_ENTRY(nvx_prefill_wide)(x, x_stride, w, y, m, n, k, silu, tile == NVX_PG_256_256 ? 256 : tile == NVX_PG_192_256 ? 192 : 128, tile == NVX_PG_128_128 ? 128 : 256, st);
#define NVX_PG(TM, TN, KS, ST, MODE) launch_prefill_gemm<TM, TN, KS, ST, 2, MODE>(x, x_stride, w, y, m, n, k, qkv, st)
    if (mode == NVX_PG_QKV) switch (tile) {
        case NVX_PG_32_128: NVX_PG(32, 128, 64, 4, NVX_PG_QKV); break;
        case NVX_PG_64_128: NVX_PG(64, 128, 64, 4, NVX_PG_QKV); break;
        case NVX_PG_96_128: NVX_PG(96, 128, 64, 4, NVX_PG_QKV); break;
        case NVX_PG_HEADS_128_128: NVX_PG(128, 128, 64, 4, NVX_PG_QKV); break;
        default: return nvx_fail(NVX_EUNSUPPORTED, "nvx_prefill_gemm: no tile %d", tile);
    } else switch (tile) {
        case NVX_PG_64_128: if (silu) NVX_PG(64, 128, 64, 4, NVX_PG_SILU); else NVX_PG(64, 128, 64, 4, NVX_PG_PLAIN); break;
        case NVX_PG_64_128_THREE: NVX_REQUIRE(silu, NVX_EUNSUPPORTED, "nvx_prefill_gemm: tile"); NVX_PG(64, 128, 64, 2, NVX_PG_SILU); break;
        case NVX_PG_96_128: if (silu) NVX_PG(96, 128, 64, 4, NVX_PG_SILU); else NVX_PG(96, 128, 64, 4, NVX_PG_PLAIN); break;
        case NVX_PG_160_128: if (silu) NVX_PG(160, 128, 64, 4, NVX_PG_SILU); else NVX_PG(160, 128, 64, 4, NVX_PG_PLAIN); break;
        case NVX_PG_192_128: if (silu) NVX_PG(192, 128, 64, 4, NVX_PG_SILU); else NVX_PG(192, 128, 64, 4, NVX_PG_PLAIN); break;
        case NVX_PG_224_128: if (silu) NVX_PG(224, 128, 64, 3, NVX_PG_SILU); else NVX_PG(224, 128, 64, 3, NVX_PG_PLAIN); break;
        case NVX_PG_64_64: if (silu) NVX_PG(64, 64, 64, 4, NVX_PG_SILU); else NVX_PG(64, 64, 64, 4, NVX_PG_PLAIN); break;
        case NVX_PG_32_64: if (silu) NVX_PG(32, 64, 128, 4, NVX_PG_SILU); else NVX_PG(32, 64, 128, 4, NVX_PG_PLAIN); break;
        case NVX_PG_96_64: NVX_REQUIRE(!silu, NVX_EUNSUPPORTED, "nvx_prefill_gemm: tile"); NVX_PG(96, 64, 64, 4, NVX_PG_PLAIN); break;
        case NVX_PG_128_64: NVX_REQUIRE(!silu, NVX_EUNSUPPORTED, "nvx_prefill_gemm: tile"); NVX_PG(128, 64, 64, 4, NVX_PG_PLAIN); break;
        case NVX_PG_160_64: NVX_REQUIRE(!silu, NVX_EUNSUPPORTED, "nvx_prefill_gemm: tile"); NVX_PG(160, 64, 64, 4, NVX_PG_PLAIN); break;
        case NVX_PG_192_64: NVX_REQUIRE(!silu, NVX_EUNSUPPORTED, "nvx_prefill_gemm: tile"); NVX_PG(192, 64, 64, 4, NVX_PG_PLAIN); break;
        case NVX_PG_32_32: NVX_REQUIRE(!silu, NVX_EUNSUPPORTED, "nvx_prefill_gemm: tile"); NVX_PG(32, 32, 128, 4, NVX_PG_PLAIN); break;
        default: return nvx_fail(NVX_EUNSUPPORTED, "nvx_prefill_gemm: no tile %d", tile);
    }
#undef NVX_PG
    return nvx_check_launch("nvx_prefill_gemm");
}
int NVX_ENTRY(nvx_prefill_gemm)(const void* x, int64_t x_stride, const void* w, void* y, int64_t m, int64_t n, int64_t k, int mode, const NvxQkvOut* qkv, hipStream_t st) {
    return prefill_gemm(0, x, x_stride, w, y, m, n, k, mode, qkv, st);
}
// one product, PLAIN or SILU, by a tile of the caller's choice (0: the rule's)
extern "C" int NVX_ENTRY(nvx_internal_prefill_gemm)(const void* x, int64_t x_stride, const void* w, void* y, int64_t m, int64_t n, int64_t k, int silu, int tile,
                                                    nvx_stream_t stream) {
    return prefill_gemm(tile, x, x_stride, w, y, m, n, k, silu ? NVX_PG_SILU : NVX_PG_PLAIN, nullptr, (hipStream_t)stream);
}
// the rule's tile
extern "C" int NVX_ENTRY(nvx_internal_prefill_tile)(int64_t m, int64_t n, int64_t k, int silu) {
    float cost;
    return prefill_gemm_rule(m, n, k, silu, n * k < (1ll << 30), cost);
}
// what becomes of one [q | k | v] projection, by a tile of the caller's choice (0: the rule's)
extern "C" int NVX_ENTRY(nvx_internal_prefill_heads)(const void* x, int64_t x_stride, const void* w, int64_t m, int64_t k, int tile, const int64_t* positions, const int64_t* slots,
                                                     const float* rope, int64_t rope_rows, int64_t n_slots, const void* q_norm, const void* k_norm, void* q, void* k_cache, void* v_cache,
                                                     int hq, int hkv, float eps, nvx_stream_t stream) {
    const NvxQkvOut out = {positions, slots, rope, rope_rows, n_slots, (const uint16_t*)q_norm, (const uint16_t*)k_norm, (uint16_t*)q, (uint16_t*)k_cache, (uint16_t*)v_cache, hq, hkv, eps};
    return prefill_gemm(tile, x, x_stride, w, nullptr, m, (int64_t)(hq + 2 * hkv) * 128, k, NVX_PG_QKV, &out, (hipStream_t)stream);
}
