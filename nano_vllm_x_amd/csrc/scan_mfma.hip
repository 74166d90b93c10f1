// The recurrences over a (key size x value size) memory per head on the matrix cores, for portions of several tokens: decay, gla and mlstm
// (see state_scan.hip for what they compute, for their phases over chunks side by side, and for single tokens and wider keys).
//
// Sixteen tokens at a time the recurrence is three small products.  With b_i the decay from the block's start to token i, w_j from token j
// to its end and d_ij from j to i:
//     O = diag(b) Q S  +  (Q K^T o d) V  (d_ij = 0 for j > i);      S <- keep S + K^T diag(w) V.
// The memory stays in the accumulators of v_mfma_f32_16x16x4_f32 from block to block: a wave keeps all key rows of 16 value columns, and an
// accumulator register is the B operand of Q S as it stands (lane group q, register r: row 16 dt + 4 q + r).  Products and sums are float32
// in every format; every factor is a product of decays, or an exponential of a difference of gate sums formed in double precision, and at
// most one, whatever the gates (no factor is ever divided out).
//   decay   one constant per head: powers of it.
//   gla     a decay per key channel and token: b and w are running products per channel, laid into the staged queries and keys; Q K^T o d is
//           formed on the vector ALU, a lane walking its key's channels forward in time (a quotient of products could overflow).
//   mlstm   log gates and a running maximum m: with u_i = F_i - m_i and g_j = i_j - F_j (F: the sum of forget gates) every factor is
//           exp(u_i + g_j) or exp(u_i - u_s).  The normaliser is carried beside the memory, one vector per head.
// A workgroup of eight waves takes one head of one sequence (or chunk) and up to 128 value columns.  64 tokens are staged at a time (LDS, 74
// KB at 64 keys: two workgroups a CU), the next 64 travel to registers meanwhile.  Bound: the matrix cores' float32 rate (36 instructions of 32
// cycles per 16 tokens and 16 columns at 64 keys).  The walk token by token that this replaces for keys of up to 128 read its staged
// rows once per token and thread and ran at 6-9 % of the vector rate.  Measured, the two
// phases over chunks, us: gla 3847 tokens of 16 heads 64 x 128 157 + 103 -> 53 + 29; mlstm the same 187 + 106 -> 62 + 33; decay 4096
// tokens of 8 such heads 58 + 38 -> 27 + 19.
#include <type_traits>

#include "scan_dev.h"

namespace NVX_NS {

constexpr int ST = 64;                 // tokens of a stage
constexpr int SC = 128;                // value columns of a workgroup
constexpr int SW = 512;                // threads

template <typename T> using Vec4 = T __attribute__((ext_vector_type(4)));

// n_ok (at most four) elements from p on, zeros behind them; `vec`: all four are there and p stands on their border
template <typename T>
__device__ __forceinline__ Vec4<T> fetch4(const T* __restrict__ p, int n_ok, bool vec) {
    if (vec && n_ok > 0) return *reinterpret_cast<const Vec4<T>*>(p);
    Vec4<T> f = {(T)0.f, (T)0.f, (T)0.f, (T)0.f};
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (k < n_ok) f[k] = p[k];
    return f;
}

template <typename A, int MODE, int PHASE, int D>
__global__ __launch_bounds__(SW, D == 64 && PHASE && sizeof(A) == 2 ? 4 : 2) void scan_mfma_kernel(ScanArgs a) {
    constexpr int LD = D + 4;                            // floats of a staged key row (16-byte pieces, rows spread over the banks)
    typedef std::conditional_t<MODE == SCAN_DECAY, float, A> VT;      // values as they came, or behind their activation
    constexpr int LV = sizeof(VT) == 4 ? SC + 4 : SC + 8;
    constexpr int NP = ST * (D / 4) / SW, NV = ST * (SC / 4) / SW;     // pieces of four elements a thread stages
    constexpr bool READS = PHASE != 1;                   // phase 1 wants the memory only
    __shared__ __align__(16) float sq[READS ? ST * LD : 4];
    __shared__ __align__(16) float sk[ST * LD];
    __shared__ __align__(16) float sa[MODE == SCAN_GLA ? ST * LD : 4];
    __shared__ __align__(16) VT sv[ST * LV];
    __shared__ __align__(16) float s_att[READS ? ST * 20 : 4];
    __shared__ float s_keep[MODE == SCAN_GLA ? 4 * D : 4];            // what a block leaves of the memory in front of it
    __shared__ float s_pow[17];                                       // decay: its powers
    __shared__ double s_u[MODE == SCAN_MLSTM ? ST : 1], s_g[MODE == SCAN_MLSTM ? ST : 1];
    __shared__ float s_b[MODE == SCAN_MLSTM ? ST : 1], s_w[MODE == SCAN_MLSTM ? ST : 1], s_m[MODE == SCAN_MLSTM ? ST : 1], s_den[MODE == SCAN_MLSTM ? ST : 1];
    __shared__ __align__(16) float s_n[MODE == SCAN_MLSTM ? 4 * D : 4];

    const int hd = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, c = lane & 15, q = lane >> 4;
    SeqSpan sp = seq_span(PHASE ? blockIdx.z / a.n_chunk_max : blockIdx.z, a.qo_indptr, a.pos0, a.state_slot);
    if (sp.slot < 0 || sp.n <= 0) return;
    if (PHASE) {
        const int64_t first = (int64_t)(blockIdx.z % a.n_chunk_max) * a.chunk;
        if (first >= sp.n) return;
        sp.q0 += first;
        sp.n = sp.n - first < a.chunk ? sp.n - first : a.chunk;
    }
    const int dim = a.dim, vdim = a.vdim, heads = a.heads;
    const int64_t at = (int64_t)(PHASE ? (int)blockIdx.z : sp.slot) * heads + hd;
    const int c0 = blockIdx.x * SC, e = c0 + wave * 16 + c;            // this lane's value column
    const bool cont = PHASE == 3 || (PHASE == 0 && sp.pos0 > 0), mine = e < vdim, works = c0 + wave * 16 < vdim;
    float* Sp = (PHASE ? a.ws : a.S) + at * dim * vdim;
    nvx_f32x4 S[D / 16];
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * dt + 4 * q + r;
            S[dt][r] = cont && mine && row < dim ? Sp[(int64_t)row * vdim + e] : 0.f;
        }

    // what a stage brings, in registers until the stage before it is done
    const A* x = (const A*)a.x;
    Vec4<A> rq[READS ? NP : 1], rk[NP], rv[NV];
    nvx_f32x4 ra[MODE == SCAN_GLA ? NP : 1];
    float gate_i = 0.f, gate_f = 0.f;
    const bool vec = a.vec != 0;
    auto ask = [&](int64_t t0) {
        const int nt = (int)(sp.n - t0 < ST ? sp.n - t0 : ST);
        const A* row0 = x + (sp.q0 + t0) * a.x_stride;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int p = threadIdx.x + i * SW, tt = p / (D / 4), d = p % (D / 4) * 4, ok = tt < nt ? dim - d : 0;
            if (READS) rq[i] = fetch4(row0 + tt * a.x_stride + a.q_off + hd * dim + d, ok, vec);
            rk[i] = fetch4(row0 + tt * a.x_stride + a.k_off + hd * dim + d, ok, vec);
            if (MODE == SCAN_GLA) {
                ra[i] = fetch4(a.alpha + (sp.q0 + t0 + tt) * heads * dim + hd * dim + d, ok, vec);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (k >= ok) ra[i][k] = 1.f;         // tokens that are not there leave the memory as it is
            }
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int p = threadIdx.x + i * SW, tt = p / (SC / 4), d = c0 + p % (SC / 4) * 4, ok = tt < nt ? vdim - d : 0;
            rv[i] = fetch4(row0 + tt * a.x_stride + a.v_off + hd * vdim + d, ok, vec);
        }
        if (MODE == SCAN_MLSTM && wave == 0) {
            const float* g = a.gates + (sp.q0 + t0 + (lane < nt ? lane : nt - 1)) * 2 * heads;
            gate_i = g[hd] + a.gate_bias[hd];
            gate_f = g[heads + hd] + a.gate_bias[heads + hd];
        }
    };
    auto act4 = [&](Vec4<A> in, float mul) {
        nvx_f32x4 v;
#pragma unroll
        for (int k = 0; k < 4; ++k) { const float z = (float)in[k]; v[k] = (MODE == SCAN_DECAY && a.act == 1 ? z * sigmoid_f(z) : z) * mul; }
        return v;
    };

    float nrm[MODE == SCAN_MLSTM ? (D + 63) / 64 : 1];                // wave 4: the normaliser's rows lane, lane + 64
    float m_run = 0.f;
    double f_all = 0.0;
    float kept = 1.f;                                                 // gla, phase 1: the product of a channel's decays
    if (MODE == SCAN_MLSTM) {
        m_run = cont ? (PHASE ? a.M_ws[at] : a.M_in[at]) : (PHASE == 1 ? -INFINITY : 0.f);
        const float* Np = PHASE ? a.N_ws : a.N_in;
#pragma unroll
        for (int i = 0; i < (int)(sizeof(nrm) / sizeof(float)); ++i) nrm[i] = cont && lane + 64 * i < dim ? Np[at * dim + lane + 64 * i] : 0.f;
    }
    if (MODE == SCAN_DECAY && threadIdx.x == 0) {
        float p = 1.f;
        for (int i = 0; i <= 16; ++i) { s_pow[i] = p; p *= a.decay[hd]; }
    }

    ask(0);
    for (int64_t t0 = 0; t0 < sp.n; t0 += ST) {
        const int nt = (int)(sp.n - t0 < ST ? sp.n - t0 : ST), n_blk = (nt + 15) / 16;
        __syncthreads();                                 // the stage before is done with
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int p = threadIdx.x + i * SW, tt = p / (D / 4), d = p % (D / 4) * 4;
            if (READS) *reinterpret_cast<nvx_f32x4*>(sq + tt * LD + d) = act4(rq[i], a.q_mul);
            *reinterpret_cast<nvx_f32x4*>(sk + tt * LD + d) = act4(rk[i], a.k_mul);
            if (MODE == SCAN_GLA) *reinterpret_cast<nvx_f32x4*>(sa + tt * LD + d) = ra[i];
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int p = threadIdx.x + i * SW, tt = p / (SC / 4), d = p % (SC / 4) * 4;
            if constexpr (MODE == SCAN_DECAY) *reinterpret_cast<nvx_f32x4*>(sv + tt * LV + d) = act4(rv[i], 1.f);
            else *reinterpret_cast<Vec4<A>*>(sv + tt * LV + d) = rv[i];
        }
        if (MODE == SCAN_MLSTM && wave == 0) {           // lane = token: gates, their sums and maxima
            const float gi = a.cap * tanhf(gate_i / a.cap), gf = logsigmoid_f(a.cap * tanhf(gate_f / a.cap));
            double F = lane < nt ? (double)gf : 0.0;
#pragma unroll
            for (int s = 1; s < 64; s <<= 1) { const double o = __shfl_up(F, s, 64); if (lane >= s) F += o; }
            const double g = (double)gi - F;
            double top = lane < nt ? g : -INFINITY;      // the largest i_j - F_j up to here
#pragma unroll
            for (int s = 1; s < 64; s <<= 1) { const double o = __shfl_up(top, s, 64); if (lane >= s && o > top) top = o; }
            if ((double)m_run > top) top = (double)m_run;
            const double u = -top;                       // F_i - m_i with m_i = F_i + max(...)
            const int last = (lane | 15) < nt ? (lane | 15) : nt - 1, front = (lane & ~15) - 1;
            const double u_end = __shfl(u, last, 64), u_front0 = __shfl(u, front < 0 ? 0 : front, 64), u_front = front < 0 ? -(double)m_run : u_front0;
            s_u[lane] = u;
            s_g[lane] = g;
            s_m[lane] = (float)(F - u);
            s_b[lane] = expf((float)(u - u_front));      // (from a start without memory: exp(-inf) = 0)
            s_w[lane] = lane < nt ? expf((float)(u_end + g)) : 0.f;
            if ((lane & 15) == 0 && lane < nt) s_keep[lane >> 4] = expf((float)(u_end - u_front));
            const double F_all = __shfl(F, nt - 1, 64);
            f_all += F_all;
            m_run = (float)(F_all - __shfl(u, nt - 1, 64));
        }
        __syncthreads();
        if (t0 + ST < sp.n) ask(t0 + ST);
        if (MODE == SCAN_DECAY && a.half) {              // rotate the pairs (m, m + half) of queries and keys by the tokens' angles
            for (int i = threadIdx.x; i < nt * a.half; i += SW) {
                const int tt = i / a.half, m = i - tt * a.half;
                const float* tr = a.turn.cos + (sp.q0 + t0 + tt) * a.turn.stride + m;
                const float co = tr[0], si = tr[a.turn.sin_off];
                float* kr = sk + tt * LD + m;
                const float u = kr[0], v = kr[a.half];
                kr[0] = u * co - v * si;
                kr[a.half] = v * co + u * si;
                if (READS) {
                    float* qr = sq + tt * LD + m;
                    const float y = qr[0], z = qr[a.half];
                    qr[0] = y * co - z * si;
                    qr[a.half] = z * co + y * si;
                }
            }
            __syncthreads();
        }
        if (MODE != SCAN_GLA && READS && wave < n_blk) { // a wave a block: Q K^T o d
            nvx_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int dt = 0; dt < D / 16; ++dt) {
                const nvx_f32x4 qa = *reinterpret_cast<const nvx_f32x4*>(sq + (16 * wave + c) * LD + 16 * dt + 4 * q);
                const nvx_f32x4 kb = *reinterpret_cast<const nvx_f32x4*>(sk + (16 * wave + c) * LD + 16 * dt + 4 * q);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[r], kb[r], acc, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {                // row (query) 4 q + r, column (key) c
                const int i = 4 * q + r;
                float d = 0.f;
                if (c <= i && 16 * wave + i < nt) {
                    if (MODE == SCAN_MLSTM) d = expf((float)(s_u[16 * wave + i] + s_g[16 * wave + c]));
                    else d = s_pow[i - c];
                }
                s_att[(16 * wave + i) * 20 + c] = c <= i && 16 * wave + i < nt ? acc[r] * d : 0.f;
            }
        }
        if (MODE == SCAN_MLSTM && wave == 4) {           // the normaliser in front of every block
            for (int b = 0; b < n_blk; ++b) {
#pragma unroll
                for (int i = 0; i < (int)(sizeof(nrm) / sizeof(float)); ++i) {
                    const int d = lane + 64 * i;
                    if (d < D) s_n[b * D + d] = nrm[i];
                    float add = 0.f;
                    if (d < D)
                        for (int j = 0; j < 16; ++j) add += s_w[16 * b + j] * sk[(16 * b + j) * LD + d];
                    nrm[i] = s_keep[b] * nrm[i] + add;
                }
            }
        }
        if (MODE == SCAN_MLSTM && READS) {
            __syncthreads();
            const int i = threadIdx.x >> 3, part = threadIdx.x & 7;    // eight lanes a token
            if (i < nt) {
                float dot = 0.f;
#pragma unroll
                for (int d = part * 4; d < D; d += 32) {
                    const nvx_f32x4 qv = *reinterpret_cast<const nvx_f32x4*>(sq + i * LD + d), nv = *reinterpret_cast<const nvx_f32x4*>(s_n + (i >> 4) * D + d);
                    dot += qv[0] * nv[0] + qv[1] * nv[1] + qv[2] * nv[2] + qv[3] * nv[3];
                }
                dot = dot * s_b[i] + s_att[i * 20 + part * 2] + s_att[i * 20 + part * 2 + 1];
                dot = group_sum<8>(dot);
                if (part == 0) s_den[i] = fmaxf(fabsf(dot), expf(-s_m[i])) + 1e-6f;
            }
            __syncthreads();
        }
        if (MODE == SCAN_GLA) {
            if (READS) {
                // eight keys of a block a wave, eight lanes a key: its channels walk forward in time
                constexpr int DL = D / 8;
                const int b = wave >> 1, half = wave & 1, j = half * 8 + (lane >> 3), d0 = (lane & 7) * DL;
                if (b < n_blk) {
                    float w[DL];
#pragma unroll
                    for (int d = 0; d < DL; ++d) w[d] = sk[(16 * b + j) * LD + d0 + d];
                    for (int i = 0; i < 16; ++i) {
                        float s = 0.f;
                        if (i >= half * 8) {             // (uniform over the wave)
                            const float* qr = sq + (16 * b + i) * LD + d0;
                            const float* ar = sa + (16 * b + i) * LD + d0;
#pragma unroll
                            for (int d = 0; d < DL; ++d) {
                                w[d] *= i > j ? ar[d] : 1.f;
                                s += qr[d] * w[d];
                            }
                            s = group_sum<8>(s);
                        }
                        if ((lane & 7) == 0) s_att[(16 * b + i) * 20 + j] = i >= j ? s : 0.f;
                    }
                }
                __syncthreads();
            }
            // the running products of a block's decays into its queries (from its start), its keys (to its end), and over all of it
            for (int i = threadIdx.x; i < n_blk * D; i += SW) {
                const int b = i / D, d = i % D;
                float p = 1.f;
                if (READS)
                    for (int t = 0; t < 16; ++t) { p *= sa[(16 * b + t) * LD + d]; sq[(16 * b + t) * LD + d] *= p; }
                p = 1.f;
                for (int t = 15; t >= 0; --t) { sk[(16 * b + t) * LD + d] *= p; p *= sa[(16 * b + t) * LD + d]; }
                s_keep[b * D + d] = p;
            }
        }
        if (MODE != SCAN_MLSTM || !READS) __syncthreads();
        if (MODE == SCAN_GLA && PHASE == 1 && blockIdx.x == 0 && (int)threadIdx.x < D)
            for (int b = 0; b < n_blk; ++b) kept *= s_keep[b * D + threadIdx.x];
        if (works) {
            for (int b = 0; b < n_blk; ++b) {
                const int nb = nt - 16 * b < 16 ? nt - 16 * b : 16;
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = (float)sv[(16 * b + 4 * q + r) * LV + wave * 16 + c];
                if (READS) {
                    nvx_f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int dt = 0; dt < D / 16; ++dt) {
                        const nvx_f32x4 qa = *reinterpret_cast<const nvx_f32x4*>(sq + (16 * b + c) * LD + 16 * dt + 4 * q);
#pragma unroll
                        for (int r = 0; r < 4; ++r) o = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[r], S[dt][r], o, 0, 0, 0);
                    }
                    if (MODE != SCAN_GLA) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) o[r] *= MODE == SCAN_MLSTM ? s_b[16 * b + 4 * q + r] : s_pow[4 * q + r + 1];
                    }
                    const nvx_f32x4 pa = *reinterpret_cast<const nvx_f32x4*>(s_att + (16 * b + c) * 20 + 4 * q);
#pragma unroll
                    for (int r = 0; r < 4; ++r) o = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[r], v[r], o, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int i = 16 * b + 4 * q + r;
                        if (i < nt && mine) {
                            const float z = MODE == SCAN_MLSTM ? o[r] / s_den[i] : o[r];
                            a.out[(sp.q0 + t0 + i) * (int64_t)heads * vdim + (int64_t)hd * vdim + e] = z;
                        }
                    }
                }
                if (PHASE == 3 && b + 1 == n_blk && t0 + ST >= sp.n) break;          // (nothing reads the memory any more)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int j = 4 * q + r;
                    if (MODE == SCAN_MLSTM) v[r] *= s_w[16 * b + j];
                    if (MODE == SCAN_DECAY) v[r] *= j < nb ? s_pow[nb - 1 - j] : 0.f;
                }
                const float keep = MODE == SCAN_MLSTM ? s_keep[b] : MODE == SCAN_DECAY ? s_pow[nb] : 1.f;
#pragma unroll
                for (int dt = 0; dt < D / 16; ++dt) {
                    if (MODE == SCAN_GLA) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) S[dt][r] *= s_keep[b * D + 16 * dt + 4 * q + r];
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r) S[dt][r] *= keep;
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        S[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(sk[(16 * b + 4 * q + r) * LD + 16 * dt + c], v[r], S[dt], 0, 0, 0);
                }
            }
        }
    }
    if (PHASE == 3) return;
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * dt + 4 * q + r;
            if (mine && row < dim) Sp[(int64_t)row * vdim + e] = S[dt][r];
        }
    if (blockIdx.x) return;
    if (MODE == SCAN_GLA && PHASE == 1 && (int)threadIdx.x < dim) a.keep_ws[at * dim + threadIdx.x] = kept;
    if (MODE == SCAN_MLSTM) {
        if (wave == 4) {
            float* Np = PHASE ? a.N_ws : a.N;
#pragma unroll
            for (int i = 0; i < (int)(sizeof(nrm) / sizeof(float)); ++i)
                if (lane + 64 * i < dim) Np[at * dim + lane + 64 * i] = nrm[i];
        }
        if (threadIdx.x == 0) {
            (PHASE ? a.M_ws : a.M)[at] = m_run;
            if (PHASE) a.F_ws[at] = (float)f_all;
        }
    }
}

}  // namespace NVX_NS

using namespace NVX_NS;

int nvx_scan_mfma_columns() { return SC; }

template <typename A, int MODE>
static void scan_mfma_launch(const ScanArgs& a, int phase, dim3 grid, hipStream_t st) {
#define NVX_SCAN_MFMA(PHASE)                                                                                      \
    do {                                                                                                          \
        if (a.dim <= 64) hipLaunchKernelGGL((scan_mfma_kernel<A, MODE, PHASE, 64>), grid, dim3(SW), 0, st, a);    \
        else hipLaunchKernelGGL((scan_mfma_kernel<A, MODE, PHASE, 128>), grid, dim3(SW), 0, st, a);               \
    } while (0)
    if (phase == 0) NVX_SCAN_MFMA(0);
    else if (phase == 1) NVX_SCAN_MFMA(1);
    else NVX_SCAN_MFMA(3);
#undef NVX_SCAN_MFMA
}

template <typename A>
static void scan_mfma_mode(const ScanArgs& a, int mode, int phase, dim3 grid, hipStream_t st) {
    if (mode == SCAN_DECAY) scan_mfma_launch<A, SCAN_DECAY>(a, phase, grid, st);
    else if (mode == SCAN_GLA) scan_mfma_launch<A, SCAN_GLA>(a, phase, grid, st);
    else scan_mfma_launch<A, SCAN_MLSTM>(a, phase, grid, st);
}

void nvx_launch_scan_mfma(const ScanArgs& in, int fmt, int mode, int phase, int64_t n_seq, hipStream_t st) {
    ScanArgs a = in;
    const dim3 grid((unsigned)((a.vdim + SC - 1) / SC), (unsigned)a.heads, (unsigned)(phase ? n_seq * a.n_chunk_max : n_seq));
    const size_t item = fmt == 2 ? 4 : 2;
    a.vec = (reinterpret_cast<uintptr_t>(a.x) & (4 * item - 1)) == 0 && ((a.x_stride | a.q_off | a.k_off | a.v_off | a.dim | a.vdim) & 3) == 0 &&
            (mode != SCAN_GLA || nvx_aligned16(a.alpha));
    NVX_FMT_CALL(fmt, scan_mfma_mode<A_>(a, mode, phase, grid, st));
}
