// y = x W^T (+ bias) for the few rows of a decode step, in the 16-bit format or as unrounded float32 sums: the projections of the models
// with per-sequence state.
//
// Such a product is one pass over W.  A workgroup of eight waves takes 16 rows of W whole (eight where there are few): every wave a strided eighth of K, 64 columns
// (a 128-byte line of every row) at a time, of W and of x, through a ring in LDS that is its own: no barrier until the waves' sums meet,
// in a fixed order.  A layer of 1024 outputs is 64 workgroups whose loads are nearly all in flight at once, where tiles that take K in
// sequence wait once per step.  Lines travel to LDS without registers; loaded straight in operand order (64 separate 16-byte requests an
// instruction, which the address unit serves one a clock) 1024 x 2048 took 5.8 us instead of 3.8.
// 16 rows, N x K, us here and the library's (and the time of W's bytes at 4.9 TB/s): 1024 x 1024 2.9, 5.9 (0.4); 4096 x 1024 4.2, 7.6 (1.7);
// 1024 x 2048 3.7, 8.2 (0.9); 2048 x 2048 4.7, 11.0 (1.7); 9216 x 2048 11.7, 16.1 (7.7); 1024 x 3072 5.3, 9.7 (1.3); 2048 x 6144 10.1, 12.0 (5.1);
// 32000 x 2048 28.8, 34.0 (26.7).  32 rows: 1024 x 2048 4.6, 8.4; 2048 x 6144 12.0, 16.6; 32000 x 1024 17, 25.
#include "fmt_dev.h"

namespace NVX_NS {

constexpr int FR_WAVES = 8;

__device__ __forceinline__ nvx_f32x4 mfma_few(nvx_u32x4 a, nvx_u32x4 b, nvx_f32x4 c, __bf16) {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}
__device__ __forceinline__ nvx_f32x4 mfma_few(nvx_u32x4 a, nvx_u32x4 b, nvx_f32x4 c, _Float16) {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}

// 64 lanes x 16 bytes from the lanes' addresses to 1 KB of LDS from a wave-uniform address on; the compiler does not count these loads, so every
// wait for them is explicit
__device__ __forceinline__ void line_to_lds(const void* g, unsigned lds) {
    const unsigned uni = (unsigned)__builtin_amdgcn_readfirstlane((int)lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "s"(uni) : "memory");
}

// the waves' sums meet in `smem` (their rings, which nobody reads any more), in a fixed order, and leave as the product's rows
template <typename A, int MT, int NT, int GLU, int WR = 16>
__device__ __forceinline__ void few_rows_end(unsigned char* smem, const nvx_f32x4 (&acc)[NT][MT], const A* __restrict__ bias, void* __restrict__ y, int f32_out,
                                             int rows, int n, int n0, float limit, float alpha, float shift) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4;
    __syncthreads();
    nvx_f32x4 (*part)[NT * MT][64] = reinterpret_cast<nvx_f32x4 (*)[NT * MT][64]>(smem);
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) part[wave][i * MT + j][lane] = acc[i][j];
    __syncthreads();
    // a lane of a tile has row l16 and the outputs 4 * quad .. 4 * quad + 3
    if constexpr (GLU != 0) {            // the projections rounded to the format, as the activation's own kernel reads them
        if (wave < MT) {
            nvx_f32x4 g = part[0][wave][lane], u = part[0][MT + wave][lane];
#pragma unroll
            for (int i = 1; i < FR_WAVES; ++i) { g += part[i][wave][lane]; u += part[i][MT + wave][lane]; }
            const int r = 16 * wave + l16;
            if (r < rows && (WR == 16 || quad < 2)) {
                typedef A vec4 __attribute__((ext_vector_type(4)));
                vec4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float gr = (float)(A)g[i], ur = (float)(A)u[i];
                    o[i] = (A)(GLU == 2 ? gelu_glu_act(gr, ur) : glu_act(gr, ur, limit, alpha, shift));
                }
                *reinterpret_cast<vec4*>((A*)y + (int64_t)r * (n / 2) + n0 + 4 * quad) = o;
            }
        }
    } else if (wave < NT * MT) {
        nvx_f32x4 s = part[0][wave][lane];
#pragma unroll
        for (int i = 1; i < FR_WAVES; ++i) s += part[i][wave][lane];
        const int r = 16 * (wave % MT) + l16, o = n0 + WR * (wave / MT) + 4 * quad;
        if (WR == 8 && quad >= 2) return;
        if (bias)
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] += (float)bias[o + i];
        if (r < rows) {
            typedef A vec4 __attribute__((ext_vector_type(4)));
            if (f32_out) *reinterpret_cast<nvx_f32x4*>((float*)y + (int64_t)r * n + o) = s;
            else *reinterpret_cast<vec4*>((A*)y + (int64_t)r * n + o) = vec4{(A)s[0], (A)s[1], (A)s[2], (A)s[3]};
        }
    }
}

// MT: tiles of 16 rows of x; DEPTH: pieces of 64 columns a wave has on their way.  k % 512 == 0, n % 16 == 0, rows <= 16 * MT.  WR: rows of w in a tile; with
// 8 the matrix instruction has each of them twice, and the second half of its results is left.
template <typename A, int MT, int NT, int DEPTH, int GLU, int WR>
__global__ __launch_bounds__(FR_WAVES * 64) void few_rows_kernel(const A* __restrict__ x, int64_t x_stride, const A* __restrict__ w,
                                                                const A* __restrict__ bias, void* __restrict__ y, int f32_out, int rows, int n, int k,
                                                                float limit, float alpha, float shift) {
    static_assert(!GLU || NT == 2, "16 gate rows and the 16 up rows beside them");
    constexpr int WL = NT * WR / 8, LOADS = WL + 2 * MT, PIECE = LOADS * 1024;      // [WR NT rows of w | 16 MT rows of x], 128 bytes each
    static_assert(DEPTH * PIECE >= MT * NT * 1024, "the sums meet in the pieces' memory");
    __shared__ __align__(16) unsigned char smem[FR_WAVES * DEPTH * PIECE];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4, n0 = blockIdx.x * WR * (GLU ? 1 : NT);
    const A* from[LOADS];                                                  // rows 8 i + lane / 8; the piece that belongs at place lane % 8
    const int r8 = lane >> 3, c = wave * 64 + ((lane & 7) ^ r8) * 8;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
        from[i] = i < WL ? w + (int64_t)(n0 + (GLU && i >= WL / 2 ? n / 2 - WR : 0) + 8 * i + r8) * k + c : x + (int64_t)min(8 * (i - WL) + r8, rows - 1) * x_stride + c;   // (rows past the last are not stored)
    const unsigned lds0 = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)smem + wave * DEPTH * PIECE;
    typedef __attribute__((address_space(3))) const nvx_u32x4 lds_u4;
    auto ask = [&](int t) {
        const unsigned at = lds0 + (unsigned)(t % DEPTH) * PIECE;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) line_to_lds(from[i] + (int64_t)t * (64 * FR_WAVES), at + i * 1024);
    };
    nvx_f32x4 acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = nvx_f32x4{0.f, 0.f, 0.f, 0.f};
    const int turns = k / (64 * FR_WAVES);
    for (int t = 0; t < DEPTH && t < turns; ++t) ask(t);
    for (int t = 0; t < turns; ++t) {
        // piece t has landed, up to DEPTH - 1 later ones need not have (only this wave reads what it asked for: no barrier)
        if (t + DEPTH <= turns) asm volatile("s_waitcnt vmcnt(%0)" : : "n"((DEPTH - 1) * LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        const unsigned at = lds0 + (unsigned)(t % DEPTH) * PIECE, w_at = at + (l16 & (WR - 1)) * 128, x_at = at + WL * 1024 + l16 * 128;
        nvx_u32x4 fw[2][NT], fx[2][MT];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const unsigned off = (unsigned)((4 * h + quad) ^ (l16 & 7)) * 16;
#pragma unroll
            for (int i = 0; i < NT; ++i) fw[h][i] = *reinterpret_cast<lds_u4*>((uintptr_t)(w_at + i * (WR * 128) + off));
#pragma unroll
            for (int j = 0; j < MT; ++j) fx[h][j] = *reinterpret_cast<lds_u4*>((uintptr_t)(x_at + j * 2048 + off));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");               // read before the place is filled again
        if (t + DEPTH < turns) ask(t + DEPTH);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j) acc[i][j] = mfma_few(fw[h][i], fx[h][j], acc[i][j], A{});
    }
    few_rows_end<A, MT, NT, GLU, WR>(smem, acc, bias, y, f32_out, rows, n, n0, limit, alpha, shift);
}

// The same with what stands in front of it: x_out = x (+ y) (+ add) (+ x_bias), h = x_out / rms(x_out) * w_norm in the format, out = h W^T.  Every
// workgroup forms all rows of h from the float32 stream: eight waves take two rows each and leave them in LDS, while eight others have the workgroup's rows of W on
// their way (loads of one wave come back in order: rows behind weights would wait for them).  Workgroup r writes row r of x_out and h (x_out is not x: others
// still read that).  k = 1024, rows <= 16: rows of 2048 take 2.4 us to come, and the
// form for them spilled; a form for narrower ones was not built.  Bound: the stream's rows come to every compute unit at some 34 bytes a clock (16 rows of 1024 with a result to
// add: 96 KB, 1.2 us), beside the weights' latency.  us, against the boundary's
// launch and the product's: 16 rows, 3072 x 1024 7.1 against 3.5 + 4.6; gated 6144 x 1024 6.8 against 3.5 + 4.8.  (With the rows loaded straight in operand order, 64
// requests of 16 bytes an instruction, and ahead of them the weights by the same waves, it came out behind the two launches: a step of 292 us took 306, now 284.)
template <typename A, int NT, int GLU>
__global__ __launch_bounds__(2 * FR_WAVES * 64) void few_rows_lead_kernel(const float* __restrict__ x, const A* __restrict__ y, int64_t y_stride,
                                                                         const float* __restrict__ add, const float* __restrict__ x_bias,
                                                                         const float* __restrict__ w_norm, float eps, float* __restrict__ x_out,
                                                                         A* __restrict__ h_out, const A* __restrict__ w, const A* __restrict__ bias,
                                                                         A* __restrict__ out, int rows, int n) {
    static_assert(!GLU || NT == 2, "16 gate rows and the 16 up rows beside them");
    constexpr int TURNS = 2, ROWS = 16, PIECE = NT * 2048, k = 64 * FR_WAVES * TURNS, PER_WAVE = ROWS / FR_WAVES;
    typedef A vec4 __attribute__((ext_vector_type(4)));
    __shared__ __align__(16) unsigned char smem[FR_WAVES * TURNS * PIECE + ROWS * k * sizeof(A)];      // pieces of w (as at few_rows_kernel) | rows of h
    unsigned char* rows_h = smem + FR_WAVES * TURNS * PIECE;
    const int wave = (threadIdx.x >> 6) & (FR_WAVES - 1), lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4, n0 = blockIdx.x * 16 * (GLU ? 1 : NT);
    if (threadIdx.x >= FR_WAVES * 64) {
        const unsigned lds0 = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)smem + wave * TURNS * PIECE;
        const int r8 = lane >> 3, c = wave * 64 + ((lane & 7) ^ r8) * 8;
#pragma unroll
        for (int t = 0; t < TURNS; ++t)
#pragma unroll
            for (int i = 0; i < 2 * NT; ++i)
                line_to_lds(w + (int64_t)(n0 + (GLU && i >= 2 ? n / 2 - 16 : 0) + 8 * i + r8) * k + c + t * (64 * FR_WAVES), lds0 + t * PIECE + i * 1024);
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        __syncthreads();
        __syncthreads();                                                   // (the two of few_rows_end)
        __syncthreads();
        return;
    }
    constexpr int P = k / 256;                                             // pieces of four numbers a lane has of a row
    nvx_f32x4 v[PER_WAVE][P], g[P];
#pragma unroll
    for (int q = 0; q < PER_WAVE; ++q) {
        const int row = wave * PER_WAVE + q;
        if (row >= rows) continue;
#pragma unroll
        for (int i = 0; i < P; ++i) v[q][i] = *reinterpret_cast<const nvx_f32x4*>(x + (int64_t)row * k + i * 256 + lane * 4);
    }
    vec4 u[PER_WAVE][P];
#pragma unroll
    for (int q = 0; q < PER_WAVE; ++q) {
        const int row = wave * PER_WAVE + q;
        if (row >= rows || !y) continue;
#pragma unroll
        for (int i = 0; i < P; ++i) u[q][i] = *reinterpret_cast<const vec4*>(y + row * y_stride + i * 256 + lane * 4);
    }
#pragma unroll
    for (int i = 0; i < P; ++i) g[i] = *reinterpret_cast<const nvx_f32x4*>(w_norm + i * 256 + lane * 4);
#pragma unroll
    for (int q = 0; q < PER_WAVE; ++q) {
        const int row = wave * PER_WAVE + q;
        if (row >= rows) continue;
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const int col = i * 256 + lane * 4;
            if (y)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[q][i][e] += (float)u[q][i][e];
            if (add) v[q][i] += *reinterpret_cast<const nvx_f32x4*>(add + (int64_t)row * k + col);
            if (x_bias) v[q][i] += *reinterpret_cast<const nvx_f32x4*>(x_bias + col);
#pragma unroll
            for (int e = 0; e < 4; ++e) ss += v[q][i][e] * v[q][i][e];
        }
        const float rn = 1.0f / sqrtf(wave_sum(ss) / (float)k + eps);
        const bool mine = (int)blockIdx.x == row;
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const int col = i * 256 + lane * 4;
            vec4 hv;
#pragma unroll
            for (int e = 0; e < 4; ++e) hv[e] = (A)(v[q][i][e] * rn * g[i][e]);
            *reinterpret_cast<vec4*>(rows_h + row * (k * 2) + ((col / 8) ^ (row & 7)) * 16 + (lane & 1) * 8) = hv;
            if (mine) {
                *reinterpret_cast<vec4*>(h_out + (int64_t)row * k + col) = hv;
                *reinterpret_cast<nvx_f32x4*>(x_out + (int64_t)row * k + col) = v[q][i];
            }
        }
    }
    __syncthreads();
    nvx_f32x4 acc[NT][1];
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[i][0] = nvx_f32x4{0.f, 0.f, 0.f, 0.f};
    const int row = min(l16, rows - 1);                                    // (rows past the last are not stored)
#pragma unroll
    for (int t = 0; t < TURNS; ++t)
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const nvx_u32x4 fx = *reinterpret_cast<const nvx_u32x4*>(rows_h + row * (k * 2) + (((t * FR_WAVES + wave) * 8 + 4 * half + quad) ^ (row & 7)) * 16);
#pragma unroll
            for (int i = 0; i < NT; ++i)
                acc[i][0] = mfma_few(*reinterpret_cast<const nvx_u32x4*>(smem + (wave * TURNS + t) * PIECE + i * 2048 + l16 * 128 + ((4 * half + quad) ^ (l16 & 7)) * 16), fx,
                                     acc[i][0], A{});
        }
    few_rows_end<A, 1, NT, GLU>(smem, acc, bias, out, 0, rows, n, n0, 0.f, 0.f, 0.f);
}

// What a workgroup waits for is its rows of w and of x, at some 34 bytes a clock for a compute unit, and 16 rows of x are as much as 16 of w.  While twice the
// workgroups still find a compute unit each, they take eight rows of w (the same sums in the same order).  us, tiles of 16 / of eight, 16 rows: 512 x 4096 5.3 / 4.7, 1024 x 2048 4.0 / 3.7,
// 2048 x 2048 5.15 / 4.7, 1024 x 3072 6.0 / 5.3, 2048 x 6144 11.4 / 10.1, gated 2048 x 1024 4.0 / 3.8, 4096 x 2048 7.0 / 6.3; one row 2048 x 2048 4.5 / 4.3; of 512 and 1024 columns nothing either way by themselves (2048 x 1024, one row 2.9 / 3.0), and a step of
// Kabidra of 1024 363 / 360; 32 rows 6.2 / 5.6; past that line 16 rows 3072 x 2048 5.6 / 6.4,
// gated 6144 x 1024 5.3 / 5.9.  (More pieces of K on their way instead, all loads of a workgroup at once: 2 to 4 % slower.)
// Beyond, 16 rows of w a workgroup leave the most workgroups for the chip; where there are more than run at once, more of them share the reads of x.  us at
// 16 rows, 16 against 64 rows of w: 9216 x 2048 11.7 / 11.9, 12288 x 2048 14.0 / 13.4, 32000 x 1024 18.2 / 14.6; at 32 rows, 16 against
// 32: 4096 x 2048 7.4 / 8.1, 6144 x 1024 7.5 / 6.1, 8192 x 4096 21.0 / 18.0.
template <typename A, int MT>
static void launch_few_rows(const void* x, int64_t x_stride, const void* w, const void* bias, void* y, int f32_out, int rows, int n, int k, int glu,
                            float limit, float alpha, float shift, hipStream_t st) {
#define NVX_FEW(N_, D_, G_, W_) hipLaunchKernelGGL((few_rows_kernel<A, MT, N_, D_, G_, W_>), dim3((unsigned)(n / (W_ * N_))), dim3(FR_WAVES * 64), 0, st, (const A*)x, x_stride, \
                                           (const A*)w, (const A*)bias, y, f32_out, rows, n, k, limit, alpha, shift)
    constexpr int CUS = 256;
    if (glu && n <= 16 * CUS) {
        if (glu == 1) NVX_FEW(2, 2, 1, 8);
        else NVX_FEW(2, 2, 2, 8);
    } else if (glu == 1) NVX_FEW(2, 2, 1, 16);
    else if (glu == 2) NVX_FEW(2, 2, 2, 16);
    else if (n >= 12288 && n % 64 == 0) NVX_FEW(4, 1, 0, 16);
    else if (MT == 2 && n > 4096 && n % 32 == 0) NVX_FEW(2, 2, 0, 16);
    else if (n <= 8 * CUS) NVX_FEW(1, 2, 0, 8);
    else NVX_FEW(1, 2, 0, 16);
#undef NVX_FEW
}

}  // namespace NVX_NS

using namespace NVX_NS;

// x (rows <= 32, k), rows x_stride elements apart; w (n, k) contiguous; bias (n) in the same format, or null; y (rows, n) contiguous, in the format or
// float32.  k a multiple of 512, n of 16.  glu 1 / 2: w is [gate | up] and y (rows, n / 2), in the format, is glu_act / gelu_glu_act of the two halves (n a
// multiple of 32, no bias); what the activation's own launch costs is saved (3 us of 8 for 16 rows of 6144 x 1024).
extern "C" int nvx_internal_few_rows(const void* x, int64_t x_stride, const void* w, const void* bias, void* y, int fmt, int f32_out, int64_t rows, int64_t n,
                                     int64_t k, int glu, float limit, float alpha, float shift, nvx_stream_t stream) {
    NVX_REQUIRE(glu >= 0 && glu <= 2 && (glu == 0 || (n % 32 == 0 && !bias && !f32_out)), NVX_EINVAL, "nvx_internal_few_rows: gated products");
    NVX_REQUIRE(x && w && y, NVX_EINVAL, "nvx_internal_few_rows: null pointer");
    NVX_REQUIRE(rows > 0 && rows <= 32 && n > 0 && n % 16 == 0 && n < (1 << 28) && k > 0 && k % 512 == 0 && k < (1 << 28) && (fmt == 0 || fmt == 1), NVX_EUNSUPPORTED,
                "nvx_internal_few_rows: sizes");
    NVX_REQUIRE(x_stride >= k && x_stride % 8 == 0 && nvx_aligned16(x) && nvx_aligned16(w) && nvx_aligned16(y), NVX_EINVAL, "nvx_internal_few_rows: alignment");
    const hipStream_t st = (hipStream_t)stream;
#define NVX_FEW_MT(A_)                                                                                                       \
    do {                                                                                                                     \
        if (rows <= 16) launch_few_rows<A_, 1>(x, x_stride, w, bias, y, f32_out, (int)rows, (int)n, (int)k, glu, limit, alpha, shift, st); \
        else launch_few_rows<A_, 2>(x, x_stride, w, bias, y, f32_out, (int)rows, (int)n, (int)k, glu, limit, alpha, shift, st); \
    } while (0)
    if (fmt == 0) NVX_FEW_MT(__bf16);
    else NVX_FEW_MT(_Float16);
#undef NVX_FEW_MT
    return nvx_check_launch("nvx_internal_few_rows");
}

// The residual sum and RMS norm in front of a product, in its launch: x, add (rows, k) and x_bias, w_norm (k) float32, y (rows, k) in the format, rows y_stride apart
// (y, add, x_bias may be null); x_out (rows, k) float32, not x; h (rows, k) and out (rows, n, or n / 2 with gelu) in the format.  rows <= 16, k 1024, gelu 0 or 1.
extern "C" int nvx_internal_few_rows_lead(const float* x, const void* y, int64_t y_stride, const float* add, const float* x_bias, const float* w_norm, float eps,
                                          float* x_out, void* h, const void* w, const void* bias, void* out, int fmt, int64_t rows, int64_t n, int64_t k, int gelu,
                                          nvx_stream_t stream) {
    NVX_REQUIRE(x && w_norm && x_out && h && w && out && x_out != x, NVX_EINVAL, "nvx_internal_few_rows_lead: null pointer, or the stream in place");
    NVX_REQUIRE(rows > 0 && rows <= 16 && k == 1024 && n < (1 << 28) && n % (gelu ? 32 : 16) == 0 && n / (gelu ? 32 : 16) >= 16 && (!gelu || !bias) &&
                    (fmt == 0 || fmt == 1), NVX_EUNSUPPORTED, "nvx_internal_few_rows_lead: sizes");
    NVX_REQUIRE((!y || (y_stride >= k && y_stride % 8 == 0)) && nvx_aligned16(x) && nvx_aligned16(y) && nvx_aligned16(add) && nvx_aligned16(x_bias) && nvx_aligned16(x_out) &&
                    nvx_aligned16(h) && nvx_aligned16(w) && nvx_aligned16(out), NVX_EINVAL, "nvx_internal_few_rows_lead: alignment");
#define NVX_LEAD(A_, NT, G)                                                                                                                                      \
    hipLaunchKernelGGL((few_rows_lead_kernel<A_, NT, G>), dim3((unsigned)(n / (G ? 32 : 16))), dim3(2 * FR_WAVES * 64), 0, (hipStream_t)stream, x, (const A_*)y, y_stride, add, \
                       x_bias, w_norm, eps, x_out, (A_*)h, (const A_*)w, (const A_*)bias, (A_*)out, (int)rows, (int)n)
    if (gelu && fmt == 0) NVX_LEAD(__bf16, 2, 2);
    else if (gelu) NVX_LEAD(_Float16, 2, 2);
    else if (fmt == 0) NVX_LEAD(__bf16, 1, 0);
    else NVX_LEAD(_Float16, 1, 0);
#undef NVX_LEAD
    return nvx_check_launch("nvx_internal_few_rows_lead");
}
