// Matrix products by tiles of up to 256 x 256 outputs of eight waves: the walk over K, for prefill_wide.hip and moe_gemm.hip.
//
// Such a product is bound by its matrix instructions (65 % of the kernel's clocks in each, at 2.0 GHz or less under full load) and, next to them, by LDS, of which
// eight waves read 1.5 bytes for every 512 operations.  So everything is dealt out evenly: a step is 64 columns of K, both operands memory -> LDS without
// registers, two or four steps on their way; in each half of a step a wave multiplies 32 columns while it reads the next 32, and one barrier a step, between the halves, says that a
// step has landed everywhere and that its predecessor may be overwritten.  Copies are asked for one between every four products: all at once they stop the
// wave that asks (15754 x 1024 x 2048: 56.2 us, dealt out 53.3); their addresses are a buffer's, so that a copy costs two scalar instructions and at most one of the
// vector's, and rows past the last read zeros.  A workgroup takes its share of the tiles without a pause: the last steps of a tile ask for the first of the next, and
// results turn around in LDS of their own.  K is in order, one chain of v_mfma_f32_16x16x32 an output, as in prefill_gemm.hip.
#pragma once
#include "nvx_dev.h"

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

// TM rows of x by TN rows of w a tile, STAGES steps on their way, WM x WN waves
template <int TM_, int TN_, int STAGES_, int WM, int WN>
struct WideTile {
    static constexpr int TM = TM_, TN = TN_, STAGES = STAGES_, KS = 64, FM = TM / WM / 16, FN = TN / WN / 16;     // columns of a step; fragments of a wave
    static constexpr int LOADS = (TM + TN) / 8 / (WM * WN), STAGE = (TM + TN) * KS * 2, EACH = 4;                  // copies of a wave a step; products between two of them
    static_assert((TM + TN) % (8 * WM * WN) == 0 && FM * FN % EACH == 0, "tile");
    static constexpr bool MIXED = TM / 8 % LOADS != 0;                     // a wave copies rows of both

    // A workgroup's tiles one behind the other, k / 64 == steps >= STAGES.  ask(i, step, to): the wave's copy i of eight rows of a step, of the tile that begin() or next()
    // placed last, to 1 KB of LDS; begin(): a tile's products begin; next(): its last copies have been asked for, the next tile's follow (behind the last tile
    // any that may be read); finish(acc): its sums, a lane's rows of x l16 of every 16 (second index) and of w 4 * quad .. of every 16 (first); whether another follows.
    template <typename Ask, typename Begin, typename Next, typename Mul, typename Finish>
    static __device__ __forceinline__ void walk(unsigned lds0, int steps, Ask ask, Begin begin, Next next, Mul mul, Finish finish) {
        const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4;
        const int wm = wave / WN, wn = wave % WN;
        nvx_f32x4 acc[FN][FM];
        typedef __attribute__((address_space(3))) const nvx_u32x4 lds_u4;
        struct Operands { nvx_u32x4 x[FM], w[FN]; };
        const unsigned xl = lds0 + (wm * FM * 16 + l16) * (KS * 2), wl = lds0 + (TM + wn * FN * 16 + l16) * (KS * 2);
        const unsigned piece[2] = {(unsigned)(quad ^ (l16 & 7)) * 16, (unsigned)((4 + quad) ^ (l16 & 7)) * 16};
        auto read = [&](int q, unsigned off, Operands& f) __attribute__((always_inline)) {
            if (q < FM) f.x[q] = *reinterpret_cast<lds_u4*>((uintptr_t)(xl + off + q * 16 * KS * 2));
            else f.w[q - FM] = *reinterpret_cast<lds_u4*>((uintptr_t)(wl + off + (q - FM) * 16 * KS * 2));
        };
        auto ask_for = [&](int i, int step, int slot) __attribute__((always_inline)) { ask(i, step, lds0 + (unsigned)slot * STAGE + (wave * LOADS + i) * 1024); };
        // half a step: `now` is multiplied, `next` read (the half of the step in `slot` that FIRST says), with FIRST the step `asked` asked for
        auto half = [&](const Operands& now, Operands& then, int slot, auto first, int asked, int ask_slot) __attribute__((always_inline)) {
            constexpr bool FIRST = decltype(first)::value;
            constexpr int READS = FM + FN, CHUNKS = FM * FN / EACH, R = CHUNKS >= 8 ? CHUNKS - 2 : CHUNKS;     // (the reads end before the products do)
            const unsigned off = piece[FIRST ? 0 : 1] + (unsigned)slot * STAGE;
#pragma unroll
            for (int i = 0; i < CHUNKS; ++i) {
#pragma unroll
                for (int q = 0; q < READS; ++q)
                    if (q * R / READS == i) read(q, off, then);
                if constexpr (FIRST) {
#pragma unroll
                    for (int q = 0; q < LOADS; ++q)
                        if (q * CHUNKS / LOADS == i) ask_for(q, asked, ask_slot);
                }
#pragma unroll
                for (int u = i * EACH; u < (i + 1) * EACH; ++u) acc[u / FM][u % FM] = mul(now.w[u / FM], now.x[u % FM], acc[u / FM][u % FM]);
                __builtin_amdgcn_sched_barrier(0);
            }
            wide_lds_wait();
            __builtin_amdgcn_sched_barrier(0);
        };
        for (int s = 0; s < STAGES; ++s)
#pragma unroll
            for (int i = 0; i < LOADS; ++i) ask_for(i, s, s);
        Operands even, odd;
        int slot = 0;
        wide_wait_for_all_but<(STAGES - 1) * LOADS>();
        __syncthreads();
#pragma unroll
        for (int q = 0; q < FM + FN; ++q) read(q, piece[0], even);
        wide_lds_wait();
        for (bool more = true; more;) {
            begin();
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int j = 0; j < FM; ++j) acc[i][j] = nvx_f32x4{0.f, 0.f, 0.f, 0.f};
            int asked = STAGES;
            for (int s = 0; s < steps; ++s) {
                half(even, odd, slot, std::false_type{}, 0, 0);
                wide_wait_for_all_but<(STAGES - 2) * LOADS>();          // the step behind this one has landed (as have, behind a tile, the stores of its results: they are younger and count too)
                __builtin_amdgcn_s_barrier();                           // everybody's part of it has, and everybody has read this one (wide_lds_wait)
                asm volatile("" : : : "memory");
                const int was = slot;
                slot = slot + 1 == STAGES ? 0 : slot + 1;
                if (asked == steps) {
                    asked = 0;
                    next();
                }
                half(odd, even, slot, std::true_type{}, asked, was);
                ++asked;
            }
            more = finish(acc);
        }
        wide_wait_for_all_but<0>();      // (nothing may still be on its way to this memory when it is another workgroup's)
    }
};

}  // namespace NVX_NS
