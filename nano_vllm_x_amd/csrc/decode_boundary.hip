// Products of a Qwen3 decode step with the residual sum and RMSNorm between two of them inside the products themselves.
//
// A norm needs whole rows, so as a kernel of its own it stands between two products and costs a launch to move a few KB.  Here the product in front of a norm takes K whole in every workgroup, so it can add the residual itself, and leaves three
// things: the new residual, the unrounded sum times the norm's weight (rounded once, as the norm's result was), and per row and 8 columns (16 from 33 rows
// on) the sum of the squares.  The product behind it adds a row's squares up and multiplies its own sums by 1 / rms: (x w / rms) W = (x w) W / rms.
// bfloat16 only: unnormed rows times a norm's weight need its exponents.  Rows of 1024 only: all four products of a layer have to be kernels of this package,
// which take weights of up to 16 MB (qwen3.py); with rows of 2048 and an inner size of 6144 gate | up is 50 MB and the library's.
//
// The products are those of few_rows.hip: eight waves share K, 64 columns (a 128-byte line of every row) at a time, through a ring in LDS that
// is each wave's own, no barrier until the waves' sums meet, in a fixed order, whatever the number of rows: linear_decode.hip's products over the rms,
// which take over from 33 rows (gate | up: 17), keep it, so a row's result is the same in every batch of up to 256.
// Bound by the launch (2 us) and one trip to memory (1 us) up to 16 rows, then by the reads of x: 64 rows of w a CU wait for their lines, so few rows of w
// a workgroup.  us of 1 / 29 / 64 / 123 / 256 rows in a graph, product and norm before and the product now: 1024 x 2048 3.2 + 2.1 / 3.6 + 2.3 / 4.1 + 2.3 /
// 4.8 + 2.4 / 5.8 + 2.4, now 3.4 / 3.8 / 4.1 / 4.9 / 5.7; 1024 x 3072 3.5 / 4.2 / 5.0 / 5.7 / 7.1, now 3.8 / 4.2 / 4.6 / 5.8 / 6.9.  A layer's four products with
// what stands between them: 22.2 / 25.6 / 30.3 / 34.2 / 42.2, now 17.7 / 22.6 / 26.3 / 31.6 / 39.7.
#include "nvx_dev.h"

namespace NVX_NS {

constexpr int DB_WAVES = 8;

// 64 lanes x 16 bytes from the lanes' addresses to 1 KB of LDS from a wave-uniform address on; the compiler does not count these loads, so every
// wait for them is explicit
__device__ __forceinline__ void db_line_to_lds(const void* g, unsigned lds) {
    const unsigned uni = (unsigned)__builtin_amdgcn_readfirstlane((int)lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "s"(uni) : "memory");
}

__device__ __forceinline__ float db_row_sum(float v) {      // over the 64 lanes, in every lane
    v = quarter_sum(v);
    v += xor16(v);
    return v + xor32(v);
}

struct DbArgs {
    const uint16_t *x, *w;          // (rows, k), (n, k)
    uint16_t* y;                    // DB_PLAIN (rows, n), DB_SILU (rows, n / 2), DB_RESIDUAL (rows, n): the new residual times the next norm's weight
    int rows, n, k;
    const float* squares;           // PLAIN, SILU: (rows up to a multiple of 32, 128), what DB_RESIDUAL with WR 8 left
    float eps;
    const uint16_t *residual, *norm_w;
    uint16_t* residual_out;
    float* squares_out;             // RESIDUAL: (rows up to a multiple of 32, sums of 16 columns, of 8 with WR 8)
};
constexpr int DB_PLAIN = 0, DB_SILU = 1, DB_RESIDUAL = 2;

// WR rows of w (SILU: half of them gate rows, half the up rows beside them) by XR rows of x (blockIdx.y: which) a workgroup; DEPTH: pieces of 64 columns
// a wave has on their way.  k % 512 == 0 (PLAIN, SILU: 1024), n % WR == 0.  8 rows of either fill half a tile of the matrix instruction: what is loaded counts, not that.
template <int WR, int XR, int DEPTH, int MODE>
__global__ __launch_bounds__(DB_WAVES * 64) void decode_boundary_kernel(const DbArgs a) {
    constexpr int NT = (WR + 15) / 16, MT = (XR + 15) / 16, HALF = MODE == DB_SILU ? WR / 2 : WR;
    static_assert(WR % 8 == 0 && XR % 8 == 0 && (MODE == DB_SILU ? WR == 32 : MODE == DB_PLAIN ? WR == 16 : true), "tiles");
    constexpr int LOADS = (WR + XR) / 8, PIECE = LOADS * 1024;             // [WR rows of w | XR rows of x], 128 bytes each
    constexpr int RING = DB_WAVES * DEPTH * PIECE, RES = (XR * WR * 2 + 1023) / 1024,
                  SIDE = MODE == DB_RESIDUAL ? RES * 1024 + 1024 : XR * 128 * 4;
    static_assert(RING >= DB_WAVES * NT * MT * 1024, "the sums meet in the pieces' memory");
    __shared__ __align__(16) unsigned char smem[RING + SIDE];
    __shared__ float scale[MT * 16];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4;
    const int n0 = blockIdx.x * HALF, r0 = blockIdx.y * XR, k = a.k, last = a.rows - 1;
    const unsigned lds0 = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)smem, side = lds0 + RING;
    // what the ends of the sums need travels first
    if constexpr (MODE == DB_RESIDUAL) {
        constexpr int P = WR / 8;       // place: row, eight columns
        if (wave < RES) db_line_to_lds(a.residual + (int64_t)min(r0 + min((wave * 64 + lane) / P, XR - 1), last) * a.n + n0 + lane % P * 8, side + wave * 1024);
        if (wave == RES) db_line_to_lds(a.norm_w + n0 + lane % P * 8, side + RES * 1024);
    } else {
        for (int i = wave; i < XR / 2; i += DB_WAVES) db_line_to_lds(a.squares + (int64_t)r0 * 128 + i * 256 + lane * 4, side + i * 1024);
    }
    const uint16_t* from[LOADS];                                           // rows 8 i + lane / 8; the piece that belongs at place lane % 8
    const int r8 = lane >> 3, c = wave * 64 + ((lane & 7) ^ r8) * 8;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
        from[i] = 8 * i < WR ? a.w + (int64_t)(n0 + (MODE == DB_SILU && 8 * i >= HALF ? a.n / 2 - HALF : 0) + 8 * i + r8) * k + c
                             : a.x + (int64_t)min(r0 + 8 * i - WR + r8, last) * k + c;                     // (rows past the last are not stored)
    const unsigned ring = lds0 + wave * DEPTH * PIECE;
    typedef __attribute__((address_space(3))) const nvx_u32x4 lds_u4;
    auto ask = [&](int t) {
        const unsigned at = ring + (unsigned)(t % DEPTH) * PIECE;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) db_line_to_lds(from[i] + (int64_t)t * (64 * DB_WAVES), at + i * 1024);
    };
    nvx_f32x4 acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = nvx_f32x4{0.f, 0.f, 0.f, 0.f};
    const int turns = k / (64 * DB_WAVES), wrow = WR < 16 ? l16 & (WR - 1) : l16, xrow = XR < 16 ? l16 & (XR - 1) : l16;
    for (int t = 0; t < DEPTH && t < turns; ++t) ask(t);
    for (int t = 0; t < turns; ++t) {
        // piece t has landed, up to DEPTH - 1 later ones need not have (only this wave reads what it asked for: no barrier)
        if (t + DEPTH <= turns) asm volatile("s_waitcnt vmcnt(%0)" : : "n"((DEPTH - 1) * LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        const unsigned at = ring + (unsigned)(t % DEPTH) * PIECE;
        nvx_u32x4 fw[2][NT], fx[2][MT];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const unsigned off = (unsigned)((2 * quad + h) ^ (l16 & 7)) * 16;     // (K within a block as linear_decode.hip takes it)
#pragma unroll
            for (int i = 0; i < NT; ++i) fw[h][i] = *reinterpret_cast<lds_u4*>((uintptr_t)(at + wrow * 128 + i * 2048 + off));
#pragma unroll
            for (int j = 0; j < MT; ++j) fx[h][j] = *reinterpret_cast<lds_u4*>((uintptr_t)(at + WR * 128 + xrow * 128 + j * 2048 + off));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");               // read before the place is filled again
        if (t + DEPTH < turns) ask(t + DEPTH);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j) acc[i][j] = mfma_16x16x32_h16(fw[h][i], fx[h][j], acc[i][j]);
    }
    __syncthreads();                                                       // (every wave's last wait was for all it asked for, `side` included)
    nvx_f32x4 (*part)[NT * MT][64] = reinterpret_cast<nvx_f32x4 (*)[NT * MT][64]>(smem);
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) part[wave][i * MT + j][lane] = acc[i][j];
    if constexpr (MODE != DB_RESIDUAL) {                                   // 1 / rms of the rows, a row a wave at a time
        typedef __attribute__((address_space(3))) const float lds_f;
#pragma unroll
        for (int j = 0; j < XR / DB_WAVES; ++j) {
            const int r = wave + DB_WAVES * j;
            const unsigned at = side + r * 512 + 8 * lane;                 // (a binary tree over the columns, as linear_decode.hip adds them)
            const float ss = db_row_sum(*reinterpret_cast<lds_f*>((uintptr_t)at) + *reinterpret_cast<lds_f*>((uintptr_t)(at + 4)));
            if (lane == 0) scale[r] = 1.0f / sqrtf(ss / (float)k + a.eps);
        }
    }
    __syncthreads();
    // a lane of a tile has row l16 and the outputs 4 * quad .. 4 * quad + 3
    if (wave >= (MODE == DB_SILU ? MT : NT * MT)) return;
    const int mt = wave % MT, r = r0 + 16 * mt + l16;
    nvx_f32x4 s = part[0][wave][lane];
#pragma unroll
    for (int i = 1; i < DB_WAVES; ++i) s += part[i][wave][lane];
    const bool live = r <= last && (XR >= 16 || l16 < XR);
    if constexpr (MODE == DB_SILU) {            // the projections rounded to the format, as the activation's own kernel reads them
        nvx_f32x4 u = part[0][MT + wave][lane];
#pragma unroll
        for (int i = 1; i < DB_WAVES; ++i) u += part[i][MT + wave][lane];
        const float inv = scale[16 * mt + xrow];
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = silu_h16(round_h16(s[i] * inv)) * round_h16(u[i] * inv);
        if (live) *reinterpret_cast<uint2*>(a.y + (int64_t)r * (a.n / 2) + n0 + 4 * quad) = make_uint2(pack_h16x2(o[0], o[1]), pack_h16x2(o[2], o[3]));
    } else if constexpr (MODE == DB_PLAIN) {
        const float inv = scale[16 * mt + xrow];
        if (live) *reinterpret_cast<uint2*>(a.y + (int64_t)r * a.n + n0 + 16 * (wave / MT) + 4 * quad) =
            make_uint2(pack_h16x2(s[0] * inv, s[1] * inv), pack_h16x2(s[2] * inv, s[3] * inv));
    } else {
        const int q = (quad & (WR / 4 - 1)) + 4 * (wave / MT);             // four columns of the WR
        const uint2 res = *reinterpret_cast<const uint2*>(smem + RING + (16 * mt + xrow) * (WR * 2) + q * 8);
        const uint2 nw = *reinterpret_cast<const uint2*>(smem + RING + RES * 1024 + q * 8);
        const float v[4] = {round_h16(s[0]) + h16lo_to_f32(res.x), round_h16(s[1]) + h16hi_to_f32(res.x), round_h16(s[2]) + h16lo_to_f32(res.y), round_h16(s[3]) + h16hi_to_f32(res.y)};
        float sq = v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        sq += xor16(sq);
        if constexpr (WR >= 16) sq += xor32(sq);
        if (live && quad < WR / 4) {
            const int64_t at = (int64_t)r * a.n + n0 + 4 * q;
            *reinterpret_cast<uint2*>(a.residual_out + at) = make_uint2(pack_h16x2(v[0], v[1]), pack_h16x2(v[2], v[3]));
            *reinterpret_cast<uint2*>(a.y + at) = make_uint2(pack_h16x2(v[0] * h16lo_to_f32(nw.x), v[1] * h16hi_to_f32(nw.x)),
                                                             pack_h16x2(v[2] * h16lo_to_f32(nw.y), v[3] * h16hi_to_f32(nw.y)));
            if (quad == 0) a.squares_out[((int64_t)r * gridDim.x + blockIdx.x) * NT + wave / MT] = sq;
        }
    }
}

}  // namespace NVX_NS

using namespace NVX_NS;

// mode 0: y (rows <= 32, n) = x w^T / rms; 1: y (rows <= 16, n / 2) = SiluAndMul of it, w = [gate | up]; both with k 1024 and squares as mode 2 leaves them.  2:
// residual_out = x w^T + residual, y = (the same unrounded) norm_w, squares (rows up to a multiple of 32, n / 8 up to 32 rows, n / 16 from there).
extern "C" int nvx_internal_decode_boundary(const void* x, const void* w, void* y, int64_t rows, int64_t n, int64_t k, int mode, float* squares, float eps,
                                            const void* residual, const void* norm_w, void* residual_out, nvx_stream_t stream) {
    NVX_REQUIRE(x && w && y && squares && (mode != 2 || (residual && norm_w && residual_out)), NVX_EINVAL, "nvx_internal_decode_boundary: null pointer");
    NVX_REQUIRE(mode >= 0 && mode <= 2 && rows > 0 && rows <= 256 && n > 0 && n < (1 << 24) && k > 0 && k < (1 << 24) && n % (mode == 1 ? 32 : 16) == 0 && k % 512 == 0 &&
                (mode == 2 || (k == 1024 && rows <= (mode == 1 ? 16 : 32))), NVX_EUNSUPPORTED,
                "nvx_internal_decode_boundary: sizes");
    NVX_REQUIRE(nvx_aligned16(x) && nvx_aligned16(w) && nvx_aligned16(y) && nvx_aligned16(squares) && nvx_aligned16(residual) && nvx_aligned16(norm_w) &&
                nvx_aligned16(residual_out), NVX_EINVAL, "nvx_internal_decode_boundary: pointers must be 16-byte aligned");
    const DbArgs a = {(const uint16_t*)x, (const uint16_t*)w, (uint16_t*)y, (int)rows, (int)n, (int)k, squares, eps, (const uint16_t*)residual,
                      (const uint16_t*)norm_w, (uint16_t*)residual_out, squares};
    const hipStream_t st = (hipStream_t)stream;
    // us, 1024 x 2048: 8 rows, 8 rows of w a workgroup 3.5, 16 of them 3.9; 29 rows, 8 by 16 rows of x 3.8, 16 by 32 4.7; 64 rows, 16 by 16 4.1, 16 by 32 4.8; 123 rows,
    // 16 by 32 4.9, 16 by 16 5.5; 160 rows, 32 by 32 5.4, 16 by 32 7.6.  6144 x 1024 with the activation, 1 row: 16 + 16 rows of w 5.0, 8 + 8 5.3
#define NVX_DB(WR_, XR_, D_, MODE_) hipLaunchKernelGGL((decode_boundary_kernel<WR_, XR_, D_, MODE_>), \
        dim3((unsigned)(n / (WR_)), (unsigned)((rows + XR_ - 1) / (XR_))), dim3(DB_WAVES * 64), 0, st, a)
    if (mode == 0) { if (rows <= 8) NVX_DB(16, 8, 2, DB_PLAIN); else if (rows <= 16) NVX_DB(16, 16, 2, DB_PLAIN); else NVX_DB(16, 32, 2, DB_PLAIN); }
    else if (mode == 1) { if (rows <= 8) NVX_DB(32, 8, 2, DB_SILU); else NVX_DB(32, 16, 2, DB_SILU); }
    else if (rows <= 8) NVX_DB(8, 8, 4, DB_RESIDUAL);
    else if (rows <= 32) NVX_DB(8, 16, 3, DB_RESIDUAL);
    else if (rows <= 64) NVX_DB(16, 16, 2, DB_RESIDUAL);
    else if (rows <= 128 || n % 32) NVX_DB(16, 32, 3, DB_RESIDUAL);
    else NVX_DB(32, 32, 2, DB_RESIDUAL);
#undef NVX_DB
    return nvx_check_launch("nvx_internal_decode_boundary");
}
