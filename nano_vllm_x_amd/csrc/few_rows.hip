// y = x W^T (+ bias) for the few rows of a decode step, in the 16-bit format or as unrounded float32 sums: the projections of the models
// with per-sequence state.
//
// Such a product is one pass over W.  A workgroup of eight waves takes 16 rows of W whole: every wave a strided eighth of K, 64 columns
// (a 128-byte line of every row) at a time, of W and of x, through a ring in LDS that is its own: no barrier until the waves' sums meet,
// in a fixed order.  A layer of 1024 outputs is 64 workgroups whose loads are nearly all in flight at once, where tiles that take K in
// sequence wait once per step.  Lines travel to LDS without registers; loaded straight in operand order (64 separate 16-byte requests an
// instruction, which the address unit serves one a clock) 1024 x 2048 took 5.8 us instead of 3.8.
// 16 rows, N x K, us here and the library's (and the time of W's bytes at 4.9 TB/s): 1024 x 1024 3.2, 5.9 (0.4); 4096 x 1024 4.2, 7.6 (1.7);
// 1024 x 2048 3.8, 8.2 (0.9); 2048 x 2048 5.0, 11.0 (1.7); 9216 x 2048 11.7, 16.1 (7.7); 1024 x 3072 4.6, 9.7 (1.3); 2048 x 6144 11.7, 12.0 (5.1);
// 32000 x 2048 28.8, 34.0 (26.7).  32 rows: 1024 x 2048 4.5, 8.4; 2048 x 6144 13.5, 16.6; 32000 x 1024 17, 25.
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

// MT: tiles of 16 rows of x; DEPTH: pieces of 64 columns a wave has on their way.  k % 512 == 0, n % 16 == 0, rows <= 16 * MT.
template <typename A, int MT, int NT, int DEPTH, int GLU>
__global__ __launch_bounds__(FR_WAVES * 64) void few_rows_kernel(const A* __restrict__ x, int64_t x_stride, const A* __restrict__ w,
                                                                const A* __restrict__ bias, void* __restrict__ y, int f32_out, int rows, int n, int k,
                                                                float limit, float alpha, float shift) {
    static_assert(!GLU || NT == 2, "16 gate rows and the 16 up rows beside them");
    constexpr int PIECE = (NT + MT) * 2048, LOADS = 2 * (NT + MT);         // [16 NT rows of w | 16 MT rows of x], 128 bytes each
    static_assert(DEPTH * PIECE >= MT * NT * 1024, "the sums meet in the pieces' memory");
    __shared__ __align__(16) unsigned char smem[FR_WAVES * DEPTH * PIECE];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4, n0 = blockIdx.x * 16 * (GLU ? 1 : NT);
    const A* from[LOADS];                                                  // rows 8 i + lane / 8; the piece that belongs at place lane % 8
    const int r8 = lane >> 3, c = wave * 64 + ((lane & 7) ^ r8) * 8;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
        from[i] = i < 2 * NT ? w + (int64_t)(n0 + (GLU && i >= 2 ? n / 2 - 16 : 0) + 8 * i + r8) * k + c : x + (int64_t)min(8 * (i - 2 * NT) + r8, rows - 1) * x_stride + c;   // (rows past the last are not stored)
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
        const unsigned at = lds0 + (unsigned)(t % DEPTH) * PIECE + l16 * 128;
        nvx_u32x4 fw[2][NT], fx[2][MT];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const unsigned off = (unsigned)((4 * h + quad) ^ (l16 & 7)) * 16;
#pragma unroll
            for (int i = 0; i < NT; ++i) fw[h][i] = *reinterpret_cast<lds_u4*>((uintptr_t)(at + i * 2048 + off));
#pragma unroll
            for (int j = 0; j < MT; ++j) fx[h][j] = *reinterpret_cast<lds_u4*>((uintptr_t)(at + (NT + j) * 2048 + off));
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
            if (r < rows) {
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
        const int r = 16 * (wave % MT) + l16, o = n0 + 16 * (wave / MT) + 4 * quad;
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

// 16 rows of w a workgroup leave the most workgroups for the chip; where there are more than run at once, more of them share the reads of x.  us at
// 16 rows, 16 against 64 rows of w: 9216 x 2048 11.7 / 11.9, 12288 x 2048 14.0 / 13.4, 32000 x 1024 18.2 / 14.6; at 32 rows, 16 against
// 32: 4096 x 2048 7.4 / 8.1, 6144 x 1024 7.5 / 6.1, 8192 x 4096 21.0 / 18.0.
template <typename A, int MT>
static void launch_few_rows(const void* x, int64_t x_stride, const void* w, const void* bias, void* y, int f32_out, int rows, int n, int k, int glu,
                            float limit, float alpha, float shift, hipStream_t st) {
#define NVX_FEW(N_, D_, G_) hipLaunchKernelGGL((few_rows_kernel<A, MT, N_, D_, G_>), dim3((unsigned)(n / (16 * N_))), dim3(FR_WAVES * 64), 0, st, (const A*)x, x_stride, \
                                           (const A*)w, (const A*)bias, y, f32_out, rows, n, k, limit, alpha, shift)
    if (glu == 1) NVX_FEW(2, 2, 1);
    else if (glu == 2) NVX_FEW(2, 2, 2);
    else if (n >= 12288 && n % 64 == 0) NVX_FEW(4, 1, 0);
    else if (MT == 2 && n > 4096 && n % 32 == 0) NVX_FEW(2, 2, 0);
    else NVX_FEW(1, 2, 0);
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
