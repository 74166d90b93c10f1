// The experts of steps of many tokens: two grouped matrix products over the (token, choice) pairs in expert order, without the pairs' numbers
// ever reaching the host.
//   up    y[r] = act(s W_gate x, s W_up x)   for row r of the expert order, x read from the token's own row (no copy into expert order), the
//         choice's weight s (where it scales the input) and the activation applied to the float32 sums;
//   down  out[r] = W_down y[r], float32.
// A workgroup of four waves takes a tile of 128 pairs of one expert and 128 rows of its weights (up: 64 gate rows and the 64 up rows beside
// them, so that a wave holds both halves of an output); which expert and tile it is comes from the experts' counts, so one launch serves
// whatever the router chose.  64 columns of both operands at a time travel memory -> LDS without registers into one of two buffers while the
// other is multiplied (v_mfma_f32_32x32x16, one barrier a step; 16-byte pieces XOR-swizzled on the global side, operand reads free of
// conflicts); 64 KB a workgroup, two a CU.  Results turn around in LDS and leave as whole rows.  Tiles are dealt so that an XCD works on
// neighbouring tiles (8 row tiles by as many weight tiles share its L2).  Bound: the CU's 64 bytes a clock from L2, at which two workgroups
// of this tile keep the matrix cores busy for at most as long as they wait.  One library product per expert and direction, with a copy into
// expert order ahead of them and the activation between, needed 16 + 3 launches and the counts on the host.
// 8192 pairs over 8 experts of 1536 x 1024: up 93 us (560 TFLOP/s), down 54 (480), the weighted sum 8.6, and with the tiles that the rule below takes (moe_wide_kernel)
// 74 and 44; the library's products with copy, activation and sum took 270 for a layer, and its counts a wait of the host.
#include "moe_dev.h"
#include "wide_dev.h"

#include <algorithm>

namespace NVX_NS {

constexpr int GT = 128;                // pairs, and weight rows, of a tile
constexpr int GK = 64;                 // columns of a step
constexpr int G_ROWS = 8;              // row tiles whose workgroups are neighbours

__device__ __forceinline__ nvx_f32x16 mfma32(nvx_u32x4 a, nvx_u32x4 b, nvx_f32x16 c, __bf16) {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}
__device__ __forceinline__ nvx_f32x16 mfma32(nvx_u32x4 a, nvx_u32x4 b, nvx_f32x16 c, _Float16) {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}

// 64 lanes x 16 bytes from the lanes' addresses to 1 KB of LDS from a wave-uniform address on.  From inline assembly: the compiler would hold
// every LDS read back until the copy has landed (it cannot tell the two buffers apart), so the wait ahead of the barrier is explicit too.
__device__ __forceinline__ void copy_to_lds(const void* g, unsigned lds) {
    const unsigned uni = (unsigned)__builtin_amdgcn_readfirstlane((int)lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "s"(uni) : "memory");
}
__device__ __forceinline__ void wait_copies() { asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); }

// x: the pairs' inputs, row src[r] / src_div (src null: row r), scale[src[r]] (or null) a factor of the sums; w: (experts, rows of UP ? 2 * n_out :
// n_out, k) row-major; out: (pairs, n_out), of type A (UP) or float32.  k is a multiple of 64, n_out of 64 (UP) or 128; n_exp <= 64.
template <typename A, bool UP>
__global__ __launch_bounds__(256, 2) void moe_group_gemm_kernel(const A* __restrict__ x, int64_t x_stride, const int32_t* __restrict__ src, int src_div,
                                                               const float* __restrict__ scale, const int32_t* __restrict__ counts, int n_exp,
                                                               const A* __restrict__ w, int k_in, int n_out, float limit, float alpha, float shift,
                                                               void* __restrict__ out) {
    __shared__ __align__(16) unsigned char smem[2 * 2 * GT * GK * 2];      // two buffers of [pairs | weight rows]
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int tiles_n = n_out / (UP ? GT / 2 : GT);
    // which tile: every lane an expert
    const int cnt = lane < n_exp ? counts[lane] : 0;
    int rows_to = cnt, tiles_to = (cnt + GT - 1) / GT;                     // (running sums, this expert's included)
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        const int a = __shfl_up(rows_to, s, 64), b = __shfl_up(tiles_to, s, 64);
        if (lane >= s) { rows_to += a; tiles_to += b; }
    }
    const int total = __shfl(tiles_to, 63, 64) * tiles_n, per = (total + 7) / 8;
    const int t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || t >= total) return;
    const int e = __popcll(__ballot(tiles_to * tiles_n <= t));
    const int before = e ? __shfl(tiles_to, e - 1, 64) : 0, row0 = e ? __shfl(rows_to, e - 1, 64) : 0, n_rows = __shfl(cnt, e, 64);
    const int m_tiles = (n_rows + GT - 1) / GT, tl = t - before * tiles_n;
    const int group = tl / (G_ROWS * tiles_n), gm = min(G_ROWS, m_tiles - group * G_ROWS), in = tl - group * G_ROWS * tiles_n;
    const int m0 = (group * G_ROWS + in % gm) * GT, tn = in / gm, n0 = tn * (UP ? GT / 2 : GT);
    const A* we = w + (int64_t)e * (UP ? 2 : 1) * n_out * k_in;

    // this lane's sources: rows 8 * (4 * wave + i) + lane / 8 of either operand; the piece that belongs at place lane % 8
    const int piece = (lane & 7) ^ (lane >> 3);
    const A* pa[4];
    const A* pb[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = (4 * wave + i) * 8 + (lane >> 3);
        const int m = row0 + min(m0 + r, n_rows - 1);                      // (rows past the expert's last repeat it and are not stored)
        pa[i] = x + (int64_t)(src ? src[m] / src_div : m) * x_stride + piece * 8;
        // up: weight rows in the order [32 gate | 32 up] for the first and for the second 32 outputs
        const int wr = UP ? ((r >> 5) & 1) * n_out + n0 + (r >> 6) * 32 + (r & 31) : n0 + r;
        pb[i] = we + (int64_t)wr * k_in + piece * 8;
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)smem;
    auto ask = [&](int step) {
        const unsigned buf = lds0 + (step & 1) * (2 * GT * GK * 2) + wave * 4096;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            copy_to_lds(pa[i] + step * GK, buf + i * 1024);
            copy_to_lds(pb[i] + step * GK, buf + GT * GK * 2 + i * 1024);
        }
    };
    const int wm = wave >> 1, wn = wave & 1, l32 = lane & 31, hi = lane >> 5;
    nvx_f32x16 acc[2][2];                                                  // [weight rows][pairs]
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    typedef __attribute__((address_space(3))) const nvx_u32x4 lds_u4;
    const int steps = k_in / GK;
    ask(0);
    for (int s = 0; s < steps; ++s) {
        wait_copies();
        __syncthreads();                                                   // step s is there, and nobody reads the other buffer any more
        if (s + 1 < steps) ask(s + 1);
        const unsigned xb = lds0 + (s & 1) * (2 * GT * GK * 2) + (wm * 64 + l32) * 128, wb = lds0 + (s & 1) * (2 * GT * GK * 2) + GT * GK * 2 + (wn * 64 + l32) * 128;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const unsigned off = (unsigned)((2 * kk + hi) ^ (lane & 7)) * 16;
            nvx_u32x4 fx[2], fw[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                fx[i] = *reinterpret_cast<lds_u4*>((uintptr_t)(xb + i * 4096 + off));
                fw[i] = *reinterpret_cast<lds_u4*>((uintptr_t)(wb + i * 4096 + off));
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = mfma32(fw[i], fx[j], acc[i][j], A{});
        }
    }
    // a lane has pair wm * 64 + 32 j + l32 and of every block of 32 weight rows those 8 q + 4 hi + 0..3: four neighbouring outputs at a time
    if constexpr (UP) {
        constexpr int NC = GT / 2, LO = NC + 8;                            // outputs of the tile; elements of a row of it in LDS
        typedef A vec4 __attribute__((ext_vector_type(4)));
        A* so = reinterpret_cast<A*>(smem);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int m = m0 + wm * 64 + 32 * j + l32;
            const float f = scale ? scale[src[row0 + min(m, n_rows - 1)]] : 1.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                vec4 v;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float g = fminf(f * acc[0][j][4 * q + r], limit), u = fminf(fmaxf(f * acc[1][j][4 * q + r], -limit), limit);
                    v[r] = (A)(g * sigmoid_f(alpha * g) * (u + shift));
                }
                *reinterpret_cast<vec4*>(so + (wm * 64 + 32 * j + l32) * LO + wn * 32 + 8 * q + 4 * hi) = v;
            }
        }
        __syncthreads();
        for (int p = threadIdx.x; p < GT * NC / 8; p += 256) {
            const int r = p / (NC / 8), c = p % (NC / 8) * 8;
            if (m0 + r < n_rows)
                *reinterpret_cast<nvx_u32x4*>((A*)out + (int64_t)(row0 + m0 + r) * n_out + n0 + c) = *reinterpret_cast<const nvx_u32x4*>(so + r * LO + c);
        }
    } else {
        constexpr int LO = GT + 4;
        float* so = reinterpret_cast<float*>(smem);                        // (64 pairs at a time)
        for (int h = 0; h < 2; ++h) {
            __syncthreads();
            if (wm == h) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const nvx_f32x4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                            *reinterpret_cast<nvx_f32x4*>(so + (32 * j + l32) * LO + wn * 64 + 32 * i + 8 * q + 4 * hi) = v;
                        }
            }
            __syncthreads();
            for (int p = threadIdx.x; p < 64 * GT / 4; p += 256) {
                const int r = p / (GT / 4), c = p % (GT / 4) * 4, m = m0 + 64 * h + r;
                if (m < n_rows) *reinterpret_cast<nvx_f32x4*>((float*)out + (int64_t)(row0 + m) * n_out + n0 + c) = *reinterpret_cast<const nvx_f32x4*>(so + r * LO + c);
            }
        }
    }
}

// The same products by tiles of TM pairs and TN rows of weights (up: 16 gate and 16 up rows in turn), with the walk of wide_dev.h.  k is a multiple of 64, of STAGES
// steps at least, UP ? 2 * n_out : n_out of TN; an expert's weights and all rows of x are under 2 GB.  Up: the rows' numbers are looked up when their
// tile is placed; down: an expert's rows lie together, and those past the last read zeros.
// Over 8 experts of 1536 x 1024, us in one trace, the small tile's kernel / here by 256 x 256, 192 x 256, 128 x 128: 8192 pairs, up 86 / 74, 83, 83, down 52 / 50, 44, 46;
// 5000 pairs 52 / 70, 59, 51 and 34 / 47, 44, 32; 3000 pairs 37 / 35, 31, 37 and 22 / 39, 33, 19; 200 pairs 18 / 33, 26, 16 and 18 / 30, 24, 14.  Of 3072 x 2048, 8192 pairs
// 280 / 245, 250, 267 and 161 / 168, 159, 148.  (A round costs more than prefill_wide.hip's: the activation in float32 functions.)
template <typename A>
struct MoeWideArgs {
    const A* x;
    int64_t x_stride;
    const int32_t* src;
    int src_div;
    const float* scale;
    const int32_t* counts;
    int n_exp;
    const A* w;
    int k, n_out;
    float limit, alpha, shift;
    void* out;
};
__device__ __forceinline__ nvx_f32x4 mfma16(nvx_u32x4 a, nvx_u32x4 b, nvx_f32x4 c, __bf16) {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}
__device__ __forceinline__ nvx_f32x4 mfma16(nvx_u32x4 a, nvx_u32x4 b, nvx_f32x4 c, _Float16) {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}
template <typename A, bool UP, int TM, int TN, int STAGES>
__global__ __launch_bounds__(512) void moe_wide_kernel(const MoeWideArgs<A> a) {
    constexpr int WN = 4, GROUP = 4;                                       // waves by the rows of w; tiles of pairs that share rows of w
    typedef WideTile<TM, TN, STAGES, 2, WN> T;
    constexpr int FM = T::FM, FN = T::FN, LOADS = T::LOADS;
    constexpr int OUT = UP ? TN / 2 : TN, WOUT = OUT / WN, P = WOUT / 8, SIDE = UP ? 8 * 16 * WOUT * 2 : 0;
    static_assert(!UP || (FN % 2 == 0 && (P & (P - 1)) == 0), "tile");
    __shared__ __align__(16) unsigned char smem[STAGES * T::STAGE + SIDE];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4;
    const int tiles_n = a.n_out / OUT;
    // every lane an expert: running sums of rows and of tiles, this expert's included
    const int cnt = lane < a.n_exp ? a.counts[lane] : 0;
    int rows_to = cnt, tiles_to = (cnt + TM - 1) / TM;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        const int r = __shfl_up(rows_to, s, 64), q = __shfl_up(tiles_to, s, 64);
        if (lane >= s) { rows_to += r; tiles_to += q; }
    }
    const int total = __builtin_amdgcn_readlane(tiles_to, 63) * tiles_n, per = (total + 7) / 8;
    const int last = min(((int)(blockIdx.x & 7) + 1) * per, total), stride = (int)(gridDim.x >> 3);
    int t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (t >= last) return;

    const unsigned x_bytes = (unsigned)(2 * a.x_stride), w_bytes = 2u * (unsigned)a.k, l8 = lane >> 3, c8 = ((lane & 7) ^ l8) * 16;
    int m0, tn, row0, n_rows;              // of the tile: its first pair and outputs, its expert's first pair and their number
    wide_buffer xb, wb;
    unsigned off[LOADS];
    auto of_x = [&](int i) __attribute__((always_inline)) { return (wave * LOADS + (T::MIXED ? i : 0)) * 8 < TM; };
    auto place = [&]() __attribute__((always_inline)) {
        const int e = __popcll(__ballot(tiles_to * tiles_n <= t));
        const int before = e ? __builtin_amdgcn_readlane(tiles_to, e - 1) : 0;
        row0 = e ? __builtin_amdgcn_readlane(rows_to, e - 1) : 0;
        n_rows = __builtin_amdgcn_readlane(cnt, e);
        const int m_tiles = (n_rows + TM - 1) / TM, tl = t - before * tiles_n;
        const int group = tl / (GROUP * tiles_n), gm = min(GROUP, m_tiles - group * GROUP), in = tl - group * GROUP * tiles_n;
        m0 = (group * GROUP + in % gm) * TM, tn = in / gm;
        if constexpr (UP) {
            xb = wide_buffer_at(a.x, 0x7fffffff);
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
                if (of_x(i)) off[i] = (unsigned)(a.src[row0 + min(m0 + (wave * LOADS + i) * 8 + (int)l8, n_rows - 1)] / a.src_div) * x_bytes + c8;
        } else xb = wide_buffer_at(a.x + (int64_t)(row0 + m0) * a.x_stride, (int64_t)(n_rows - 1 - m0) * x_bytes + 2 * a.k);
        wb = wide_buffer_at(a.w + ((int64_t)e * (UP ? 2 : 1) * a.n_out + (int64_t)tn * OUT) * a.k, 0x7fffffff);
    };
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = (wave * LOADS + i) * 8, rw = row - TM;
        off[i] = of_x(i) ? (row + l8) * x_bytes + c8 : ((UP ? (rw >> 4 & 1) * a.n_out + (rw >> 5) * 16 + (rw & 15) : rw) + l8) * w_bytes + c8;
    }
    auto ask = [&](int i, int step, unsigned to) __attribute__((always_inline)) { wide_to_lds(of_x(i) ? xb : wb, off[i], (unsigned)step * (T::KS * 2), to); };
    const int wm = wave / WN, wn = wave % WN;
    int m_now = 0, tn_now = 0, row_now = 0, rows_now = 0;
    auto finish = [&](nvx_f32x4 (&acc)[FN][FM]) __attribute__((always_inline)) {
        const int r0 = m_now + wm * FM * 16;
        if constexpr (UP) {
            float f[FM];
#pragma unroll
            for (int j = 0; j < FM; ++j) f[j] = a.scale ? a.scale[a.src[row_now + min(r0 + j * 16 + l16, rows_now - 1)]] : 1.0f;
            typedef A vec4 __attribute__((ext_vector_type(4)));
            unsigned char* so = smem + STAGES * T::STAGE + wave * 16 * WOUT * 2;       // a wave turns 16 rows around at a time, in memory of its own
#pragma unroll
            for (int j = 0; j < FM; ++j) {
#pragma unroll
                for (int i = 0; i < FN; i += 2) {
                    vec4 v;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float g = fminf(f[j] * acc[i][j][r], a.limit), u = fminf(fmaxf(f[j] * acc[i + 1][j][r], -a.limit), a.limit);
                        v[r] = (A)(g * sigmoid_f(a.alpha * g) * (u + a.shift));
                    }
                    *reinterpret_cast<vec4*>(so + l16 * (WOUT * 2) + (((i + (quad >> 1)) ^ (l16 & (P - 1))) * 16) + (quad & 1) * 8) = v;
                }
                wide_lds_wait();
#pragma unroll
                for (int p = 0; p < (16 * P + 63) / 64; ++p) {
                    const int r = (p * 64 + lane) / P, c = lane % P, m = r0 + j * 16 + r;
                    if (r < 16 && m < rows_now)
                        *reinterpret_cast<nvx_u32x4*>((A*)a.out + (int64_t)(row_now + m) * a.n_out + tn_now * OUT + wn * WOUT + c * 8) =
                            *reinterpret_cast<const nvx_u32x4*>(so + r * (WOUT * 2) + ((c ^ (r & (P - 1))) * 16));
                }
                wide_lds_wait();
            }
        } else {
#pragma unroll
            for (int j = 0; j < FM; ++j) {
                const int m = r0 + j * 16 + l16;
                float* at = (float*)a.out + (int64_t)(row_now + m) * a.n_out + tn_now * OUT + wn * WOUT + 4 * quad;
                if (m < rows_now)
#pragma unroll
                    for (int i = 0; i < FN; ++i) *reinterpret_cast<nvx_f32x4*>(at + 16 * i) = acc[i][j];
            }
        }
        return t < last;
    };
    place();
    T::walk((unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)smem, a.k / T::KS, ask,
            [&]() __attribute__((always_inline)) { m_now = m0, tn_now = tn, row_now = row0, rows_now = n_rows; },
            [&]() __attribute__((always_inline)) {
                t += stride;
                if (t < last) place();
            },
            [](nvx_u32x4 w, nvx_u32x4 x, nvx_f32x4 c) __attribute__((always_inline)) { return mfma16(w, x, c, A{}); }, finish);
}

// out[t] = sum_k wts[t * top + k] * o[dst[t * top + k]]   (wts == null: ones), four columns a thread.  A choice of an expert that does not exist
// (dst < 0) makes its token's result NaN: nothing on this path reads the choices on the host, and a number would pass for a result.
template <typename A>
__global__ __launch_bounds__(256) void moe_pair_gather_kernel(const float* __restrict__ o, const int64_t* __restrict__ dst, const float* __restrict__ wts,
                                                             int top, A* __restrict__ out, int64_t n, int width4) {
    typedef A vec4 __attribute__((ext_vector_type(4)));
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int64_t t = i / width4;
    const int c = (int)(i % width4) * 4;
    nvx_f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < top; ++k) {
        const float f = wts ? wts[t * top + k] : 1.0f;
        const int64_t at = dst[t * top + k];
        nvx_f32x4 v = {NAN, NAN, NAN, NAN};
        if (at >= 0) v = *reinterpret_cast<const nvx_f32x4*>(o + at * (int64_t)width4 * 4 + c);
        for (int r = 0; r < 4; ++r) sum[r] += f * v[r];
    }
    *reinterpret_cast<vec4*>(out + t * (int64_t)width4 * 4 + c) = vec4{(A)sum[0], (A)sum[1], (A)sum[2], (A)sum[3]};
}

}  // namespace NVX_NS

using namespace NVX_NS;

bool nvx_moe_grouped_fits(int fmt, int64_t n_exp, int64_t width, int64_t ff) {
    return fmt < 2 && n_exp <= 63 && width % GT == 0 && ff % 64 == 0;
}

template <typename A, bool UP, int TM, int TN, int STAGES>
static void launch_moe_wide(const MoeWideArgs<A>& a, int64_t m_tiles, hipStream_t st) {
    const int64_t tiles = m_tiles * (a.n_out / (UP ? TN / 2 : TN));
    hipLaunchKernelGGL((moe_wide_kernel<A, UP, TM, TN, STAGES>), dim3((unsigned)(tiles < 256 ? (tiles + 7) / 8 * 8 : 256)), dim3(512), 0, st, a);      // (a workgroup a CU)
}

enum { MOE_BY_RULE, MOE_256_256, MOE_192_256, MOE_128_128, MOE_FOUR_WAVES };      // tiles of pairs x rows of weights: of the wide walk, or the kernel of four waves
static const struct { int m, n, slots; float us; } MOE_TILES[] = {{256, 256, 256, 30.f}, {192, 256, 256, 28.f}, {128, 128, 256, 10.8f}, {GT, GT, 512, 21.f}};      // workgroups that run at once; us of a round of them over 1024 columns

// Which tile a product takes (n rows of weights an expert, k columns): the fewest rounds of workgroups times what a round costs (of the kernel of four waves, two a CU: 0.55 of that
// where a CU has one).  How many tiles the pairs make the counts decide, which the host does not know: the more of experts alike and of an expert's last tile
// half full for the wide tiles, whose round too many is the dearer, and the mean for the other.  us of the mixture, the tile above / four waves, where the estimate
// of half-full tiles alone went wrong: up products of 3200 pairs over 8 experts of 1536 x 1024 (192 x 256: 24 tiles of pairs, not 20) 83 / 71, 3072 x 2048 231 / 207,
// 12 000 over 60 of 1024 x 512 149 / 135.  Of 360 products measured (65 to 20 000 tokens, 2 to 63 experts, columns of 256 to 4096) four are slower than four waves, by 2 % of the mixture at most.
static int moe_tile_rule(int64_t pairs, int64_t n_exp, int64_t n, int64_t k, bool fits) {
    const int64_t live = n_exp < pairs ? n_exp : pairs;      // (experts that may have pairs)
    int best = MOE_FOUR_WAVES;
    float least = 0.f;
    for (int i = fits ? 0 : 3; i < 4; ++i) {
        const auto& t = MOE_TILES[i];
        if (i < 3 && n % t.n) continue;
        const int64_t half = std::max((2 * pairs / t.m + live) / 2, live), alike = live * ((pairs + live * t.m - 1) / (live * t.m));
        const int64_t tiles = (i == 3 ? (half + alike) / 2 : std::max(half, alike)) * ((n + t.n - 1) / t.n);
        const float cost = t.us * (i == 3 && tiles <= 256 ? 0.55f : (float)((tiles + t.slots - 1) / t.slots));
        if (best == MOE_FOUR_WAVES || cost < least) best = MOE_256_256 + i, least = cost;
    }
    return best;
}

// One of the two products, by a tile of MOE_* that fits (BY_RULE: the rule's).
template <typename A, bool UP>
static int launch_moe_product(const MoeWideArgs<A>& a, int64_t pairs, int64_t n_tok, int tile, hipStream_t st) {
    const int64_t n = UP ? 2 * (int64_t)a.n_out : a.n_out, live = a.n_exp < pairs ? a.n_exp : pairs;
    auto most = [&](int64_t tm) { return pairs / tm + live; };                                           // as many tiles as the counts can ask for
    const bool fits = a.k >= 256 && a.x_stride < (1 << 21) && n_tok * a.x_stride < (1ll << 30) && n * a.k < (1ll << 30);
    if (tile == MOE_BY_RULE) tile = moe_tile_rule(pairs, a.n_exp, n, a.k, fits);
    NVX_REQUIRE(tile == MOE_FOUR_WAVES || (tile >= MOE_256_256 && tile <= MOE_128_128 && fits && n % MOE_TILES[tile - 1].n == 0), NVX_EUNSUPPORTED, "nvx_moe_expert_rows: tile %d", tile);
    if (tile == MOE_256_256) launch_moe_wide<A, UP, 256, 256, 2>(a, most(256), st);
    else if (tile == MOE_192_256) launch_moe_wide<A, UP, 192, 256, 2>(a, most(192), st);
    else if (tile == MOE_128_128) launch_moe_wide<A, UP, 128, 128, 4>(a, most(128), st);
    else hipLaunchKernelGGL((moe_group_gemm_kernel<A, UP>), dim3((unsigned)((most(GT) * (a.n_out / (UP ? GT / 2 : GT)) + 7) / 8 * 8)), dim3(256), 0, st, a.x, a.x_stride, a.src,
                            a.src_div, a.scale, a.counts, a.n_exp, a.w, a.k, a.n_out, a.limit, a.alpha, a.shift, a.out);
    return nvx_check_launch("nvx_moe_expert_rows");
}

// The whole mixture (see nvx_moe_expert_rows) for a step of many tokens; ws as there.  The pairs' order is made here too.
static int moe_grouped(const void* h, int64_t h_stride, int fmt, const int32_t* idx, const float* wts, int64_t top, const void* w_gu, const void* w_d,
                       int64_t n_exp, float limit, float alpha, float shift, int weight_out, float* ws, void* out, int64_t n_tok, int64_t width, int64_t ff,
                       int up_tile, int down_tile, const NvxMoeEnd* end, hipStream_t st) {
    const int64_t pairs = n_tok * top;
    // ws: n_tok * top * (width + ff) floats = the pairs' results (float32), their hidden rows (16 bits), then the order: its counts, source and
    // place of every pair (12 bytes a pair and 256: they fit in the half of the hidden rows that 16 bits leave, 2 * ff >= 128 bytes a pair)
    float* o = ws;
    char* y = reinterpret_cast<char*>(ws + pairs * width);
    int64_t* dst = reinterpret_cast<int64_t*>(y + pairs * ff * 2);
    int32_t* src = reinterpret_cast<int32_t*>(dst + pairs);
    int32_t* counts = src + pairs;
    if (const int rc = nvx_moe_order_pairs(idx, pairs, n_exp, dst, src, counts, st)) return rc;
    const int64_t m_tiles = pairs / GT + (n_exp < pairs ? n_exp : pairs);
    NVX_REQUIRE(m_tiles * (ff / (GT / 2)) < (1ll << 30) && m_tiles * (width / GT) < (1ll << 30), NVX_EINVAL, "nvx_moe_expert_rows: too many tiles");
#define NVX_GROUPED(A_)                                                                                                                            \
    do {                                                                                                                                           \
        if (const int rc = launch_moe_product<A_, true>({(const A_*)h, h_stride, src, (int)top, weight_out ? (const float*)nullptr : wts, counts, (int)n_exp,         \
                                      (const A_*)w_gu, (int)width, (int)ff, limit, alpha, shift, (void*)y}, pairs, n_tok, up_tile, st)) return rc; \
        if (const int rc = launch_moe_product<A_, false>({(const A_*)y, ff, (const int32_t*)nullptr, 1, (const float*)nullptr, counts, (int)n_exp, (const A_*)w_d,    \
                                       (int)ff, (int)width, limit, alpha, shift, (void*)o}, pairs, pairs, down_tile, st)) return rc; \
        if (end) return nvx_pairs_postnorm(fmt, (const float*)o, dst, weight_out ? wts : (const float*)nullptr, top, *end, n_tok, width, st);        \
        hipLaunchKernelGGL(moe_pair_gather_kernel<A_>, dim3((unsigned)((n_tok * (width / 4) + 255) / 256)), dim3(256), 0, st, (const float*)o,     \
                           (const int64_t*)dst, weight_out ? wts : (const float*)nullptr, (int)top, (A_*)out, n_tok * (width / 4), (int)(width / 4)); \
    } while (0)
    if (fmt == 0) NVX_GROUPED(__bf16);
    else NVX_GROUPED(_Float16);
#undef NVX_GROUPED
    return nvx_check_launch("nvx_moe_expert_rows");
}

int nvx_moe_grouped(const void* h, int64_t h_stride, int fmt, const int32_t* idx, const float* wts, int64_t top, const void* w_gu, const void* w_d,
                    int64_t n_exp, float limit, float alpha, float shift, int weight_out, float* ws, void* out, int64_t n_tok, int64_t width, int64_t ff,
                    const NvxMoeEnd* end, hipStream_t st) {
    return moe_grouped(h, h_stride, fmt, idx, wts, top, w_gu, w_d, n_exp, limit, alpha, shift, weight_out, ws, out, n_tok, width, ff, MOE_BY_RULE, MOE_BY_RULE, end, st);
}

// The same with tiles of the caller's choice (0: the rule's), and the rule itself for sizes and layouts that the wide walk reads.
extern "C" int nvx_internal_moe_grouped(const void* h, int64_t h_stride, int fmt, const int32_t* idx, const float* wts, int64_t top, const void* w_gu,
                                        const void* w_d, int64_t n_exp, float limit, float alpha, float shift, int weight_out, float* ws, void* out,
                                        int64_t n_tok, int64_t width, int64_t ff, int up_tile, int down_tile, nvx_stream_t stream) {
    NVX_REQUIRE(nvx_moe_grouped_fits(fmt, n_exp, width, ff) && n_tok > 0 && n_tok <= 65535 && top > 0 && n_tok * top < (1ll << 31) && n_exp > 0 && h_stride >= width && h_stride % 8 == 0,
                NVX_EUNSUPPORTED, "nvx_internal_moe_grouped: sizes");
    NVX_REQUIRE(h && idx && wts && w_gu && w_d && ws && out && nvx_aligned16(h) && nvx_aligned16(w_gu) && nvx_aligned16(w_d) && nvx_aligned16(ws) && nvx_aligned16(out), NVX_EINVAL,
                "nvx_internal_moe_grouped: pointers must be 16-byte aligned");
    return moe_grouped(h, h_stride, fmt, idx, wts, top, w_gu, w_d, n_exp, limit, alpha, shift, weight_out, ws, out, n_tok, width, ff, up_tile, down_tile, nullptr, (hipStream_t)stream);
}
extern "C" int nvx_internal_moe_tile(int64_t pairs, int64_t n_exp, int64_t n, int64_t k) { return moe_tile_rule(pairs, n_exp, n, k, k >= 256); }
