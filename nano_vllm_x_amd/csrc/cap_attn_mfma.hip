// nvx_softcap_attn (cap_attn.hip says what it computes) on the matrix cores for steps of many tokens in a 16-bit format with heads of 128.
//
// A workgroup of four waves takes G query heads of one key/value head and 128 / G query tokens of one sequence; each wave owns 32 tokens of
// one head.  Keys are walked in tiles of 64: a tile's rows travel cache -> LDS without registers into one of two buffers while the other is
// computed, their slot ids one tile further ahead, one barrier a tile; every row fetched serves all four waves.
//   S^T (64 keys x 32 queries) = K Q^T             v_mfma_f32_32x32x16: a query's scores lie in one pair of lanes;
//   scale, cap, penalty, key norm, mask, running maximum and sum: float32 per lane, one exchange between the two lanes of a pair;
//   O^T (128 x 32 queries) += V^T P^T              v_mfma_f32_32x32x16, V^T by the LDS transpose read; P stays float32 up to here and enters
//       as hi + lo, which keeps 16 bits of it.
// Row pieces of 16 bytes are swizzled on the global side by the key's number with its bit pairs exchanged: sixteen neighbouring keys then put a
// piece at sixteen places (the products' reads of K) and four neighbouring ones four pieces apart (the transpose read of V), so tied keys and
// values are one tile.  Blocks are taken longest first over all sequences (up to 64 of them; then sequence by sequence), and where the whole
// step fits the chip at two workgroups a CU, the second one of a CU is the short counterpart of its first.
// The kernel that took 64 tokens of one head a workgroup, its keys from memory to registers by every wave, its values transposed by scalar LDS
// writes and two barriers for 32 keys, ran at 4 us a tile: 4 x 1024 tokens, 16 / 8 heads: window 512 and
// distance penalty in turn 139 -> 56 us; tied in chunks of 512, 3847 tokens: 88 -> 37.  Bound: issue slots (48 MFMAs and about 500 vector instructions a wave and
// tile) and, on short sequences, what a workgroup does once.
#include <type_traits>

#include "cap_attn_dev.h"

namespace NVX_NS {

constexpr int PT_K = 64;                                  // keys of a tile
constexpr int PT_ROW = 256;                               // bytes of a head's row

typedef __attribute__((ext_vector_type(4))) short pt_s16x4;
typedef __attribute__((address_space(3))) pt_s16x4 pt_lds_s16x4;
typedef __attribute__((address_space(3))) const nvx_u32x4 pt_lds_u4;
typedef __attribute__((address_space(3))) const nvx_f32x4 pt_lds_f4;
typedef __attribute__((address_space(3))) const int pt_lds_i32;

__device__ __forceinline__ nvx_f32x16 pt_mfma(nvx_u32x4 a, nvx_u32x4 b, nvx_f32x16 c, __bf16) {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}
__device__ __forceinline__ nvx_f32x16 pt_mfma(nvx_u32x4 a, nvx_u32x4 b, nvx_f32x16 c, _Float16) {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
}
// Copies memory -> LDS: 64 lanes' addresses to consecutive places from a wave-uniform address on.  From inline assembly, with the wait
// ahead of the barrier that publishes a tile: the compiler cannot tell the two buffers apart and would hold every LDS read back.
__device__ __forceinline__ void pt_copy16(const void* g, unsigned lds) {
    const unsigned uni = (unsigned)__builtin_amdgcn_readfirstlane((int)lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "s"(uni) : "memory");
}
__device__ __forceinline__ void pt_copy4(const void* g, unsigned lds) {
    const unsigned uni = (unsigned)__builtin_amdgcn_readfirstlane((int)lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(g), "s"(uni) : "memory");
}
__device__ __forceinline__ void pt_wait() { asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); }
__device__ __forceinline__ unsigned pt_swizzle(unsigned key) { return ((key & 3u) << 2) | ((key >> 2) & 3u); }

// Which sequence and which of its blocks of `per` tokens the block number t of the step is (b < 0: none).  Every wave finds out for itself.
__device__ __forceinline__ void pt_block_of(int t, int heads_x, const int32_t* __restrict__ qo_indptr, int n_seq, int per, int* seq, int* blk) {
    const int lane = threadIdx.x & 63;
    *seq = -1;
    *blk = 0;
    if (n_seq <= 64) {
        const int nb = lane < n_seq ? (qo_indptr[lane + 1] - qo_indptr[lane] + per - 1) / per : 0;
        auto blocks_from = [&](int level) {                                // blocks whose number in their sequence is >= level
            int v = nb > level ? nb - level : 0;
#pragma unroll
            for (int s = 1; s < 64; s <<= 1) v += __shfl_xor(v, s, 64);
            return v;
        };
        const int total = blocks_from(0);
        if (t >= total) return;
        const int pair = 256 / heads_x;                                    // blocks that give every CU one workgroup
        if (t >= pair && total <= 2 * pair) t = pair + (total - 1 - t);
        int lo = 0, hi = nb;                                               // the largest level with more than t blocks from it on
#pragma unroll
        for (int s = 1; s < 64; s <<= 1) hi = max(hi, __shfl_xor(hi, s, 64));
        while (hi - lo > 1) {
            const int mid = (lo + hi) / 2;
            if (blocks_from(mid) > t) lo = mid;
            else hi = mid;
        }
        const uint64_t there = __ballot(nb > lo);                          // sequences that have a block of this number
        int k = t - blocks_from(lo + 1);
        uint64_t m = there;
        while (k--) m &= m - 1;
        *seq = __ffsll((unsigned long long)m) - 1;
        *blk = lo;
        return;
    }
    int before = 0;
    for (int b0 = 0; b0 < n_seq; b0 += 64) {
        const int nb = b0 + lane < n_seq ? (qo_indptr[b0 + lane + 1] - qo_indptr[b0 + lane] + per - 1) / per : 0;
        int upto = nb;
#pragma unroll
        for (int s = 1; s < 64; s <<= 1) { const int o = __shfl_up(upto, s, 64); if (lane >= s) upto += o; }
        const int all = __shfl(upto, 63, 64);
        if (t < before + all) {
            const int k = __popcll(__ballot(before + upto <= t));
            const int end = __shfl(upto, k, 64) + before;
            *seq = b0 + k;
            *blk = end - 1 - t;                                            // its last block first
            return;
        }
        before += all;
    }
}

template <typename A, int G, bool TIED>
__global__ __launch_bounds__(256, 2) void softcap_attn_rows32_kernel(CapAttnArgs a) {
    constexpr int POSB = 4 / G, QPOS = 32 * POSB;
    constexpr unsigned BUF = (TIED ? 1 : 2) * PT_K * PT_ROW, IDS = PT_K * 4;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];   // two tiles, two lists of ids, two of key norms; at the end the read-out
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    int b, qblk;
    pt_block_of((int)blockIdx.y, (int)gridDim.x, a.qo_indptr, a.n_seq, QPOS, &b, &qblk);
    if (b < 0) return;
    b = __builtin_amdgcn_readfirstlane(b);
    qblk = __builtin_amdgcn_readfirstlane(qblk);
    const int per_kv = a.heads / a.kv_heads, groups = per_kv / G;
    const int kvh = blockIdx.x / groups, hd = kvh * per_kv + (blockIdx.x % groups) * G + wave % G, pb = wave / G;
    const int q0 = a.qo_indptr[b], q_n = a.qo_indptr[b + 1] - q0, qs = qblk * QPOS;
    const int rows_here = q_n - qs < QPOS ? q_n - qs : QPOS;
    const int pos_first = a.kv_len[b] - q_n + qs;                            // position of the block's first query
    const int hi = pos_first + rows_here;                                    // keys [lo, hi) are seen by some query of the block
    const int lo = first_seen(pos_first, a.window, a.chunk);
    const int32_t* slots = a.kv_indices + a.kv_start[b];
    const int row = pb * 32 + l32, pos = pos_first + row;
    const int q_lo = pos_first + pb * 32, q_hi = q_lo + 31, w_hi = q_hi + 1 < hi ? q_hi + 1 : hi;       // this wave's queries see [w_lo, w_hi)
    const int w_lo = first_seen(q_lo, a.window, a.chunk), my_lo = first_seen(pos, a.window, a.chunk);
    const bool wave_on = pb * 32 < rows_here;
    nvx_u32x4 qf[8];                                                         // dims 16 ks + 8 half .. + 7 of the lane's query
    {
        const A* qr = (const A*)a.q + ((int64_t)q0 + qs + (row < rows_here ? row : rows_here - 1)) * a.heads * 128 + (int64_t)hd * 128 + 8 * half;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) qf[ks] = *reinterpret_cast<const nvx_u32x4*>(qr + 16 * ks);
    }
    const float sink_score = a.sinks ? a.sinks[hd] : a.sink_score;
    constexpr float LOG2E = 1.4426950408889634f;
    // scores in the log2 domain, as in the tile kernel of cap_attn.hip
    const float k_lin = a.cap > 0.f ? 2.0f * a.scale * LOG2E / a.cap : a.scale * LOG2E, k_cap = a.cap * LOG2E;
    const float pen_a = a.r1 ? a.r1[hd] : 0.f, pen_b = a.r1 ? a.r2[hd] : 0.f, slope2 = a.slopes ? a.slopes[hd] * LOG2E : 0.f;
    nvx_f32x16 o_acc[4];
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[d][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    const int j_begin = lo & ~(PT_K - 1);
    // tiles of kept keys in front of the window's first tile, then the window's
    const int kept_tiles = ((a.keep < j_begin ? a.keep : j_begin) + PT_K - 1) / PT_K, n_tiles = kept_tiles + (hi - j_begin + PT_K - 1) / PT_K;
    auto tile_at = [&](int i) { return i < kept_tiles ? i * PT_K : j_begin + (i - kept_tiles) * PT_K; };
    const int place = tid & 15, krow0 = tid >> 4;                            // a pass moves 16 rows, 16 lanes a row
    const unsigned swz = pt_swizzle((unsigned)krow0);
    const unsigned char* kg = (const unsigned char*)a.k_cache + (int64_t)kvh * PT_ROW + ((unsigned)(place ^ swz) << 4);
    const unsigned char* vg = (const unsigned char*)a.v_cache + (int64_t)kvh * PT_ROW + ((unsigned)(place ^ swz) << 4);
    const int64_t row_bytes = (int64_t)a.kv_heads * PT_ROW;
    const unsigned lds0 = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)smem;
    const unsigned ids_at = lds0 + 2 * BUF, rn_at = ids_at + 2 * IDS;
    auto ask_ids = [&](int i) {                                              // by wave 0; a key past the end repeats the last and is masked
        const int j = tile_at(i) + lane;
        pt_copy4(slots + (j < hi ? j : hi - 1), ids_at + (i & 1) * IDS);
    };
    auto ask_rows = [&](int i) {
        const unsigned ids = ids_at + (i & 1) * IDS, dst = lds0 + (i & 1) * BUF + (unsigned)__builtin_amdgcn_readfirstlane(wave * 4 * PT_ROW);
        int id[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) id[p] = *reinterpret_cast<pt_lds_i32*>((uintptr_t)(ids + 4 * (krow0 + 16 * p)));
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            pt_copy16(kg + id[p] * row_bytes, dst + p * 16 * PT_ROW);
            if (!TIED) pt_copy16(vg + id[p] * row_bytes, dst + PT_K * PT_ROW + p * 16 * PT_ROW);
        }
        if (TIED && wave == 3) {                                             // the keys' reciprocal root mean squares
            const int64_t slot = *reinterpret_cast<pt_lds_i32*>((uintptr_t)(ids + 4 * lane));
            pt_copy4(a.k_rn + slot * a.kv_heads + kvh, rn_at + (i & 1) * IDS);
        }
    };
    const unsigned k_lane = l32 * PT_ROW + ((half ^ pt_swizzle(l32 & 15)) << 4);
    const unsigned v_lane = [&] {
        const unsigned grp = lane >> 4, i16 = lane & 15, r = 4 * half + (i16 >> 2), piece = 2 * (grp & 1) + ((i16 & 3) >> 1);
        return r * PT_ROW + ((piece ^ pt_swizzle(r)) << 4) + 8 * (i16 & 1);
    }();
    if (wave == 0) {
        ask_ids(0);
        if (n_tiles > 1) ask_ids(1);
    }
    pt_wait();
    __syncthreads();
    ask_rows(0);                                                             // the first two tiles travel together
    if (n_tiles > 1) ask_rows(1);
    pt_wait();
    __syncthreads();
    for (int it = 0; it < n_tiles; ++it) {
        const int j0 = tile_at(it);
        if (it + 1 < n_tiles) {                                              // the other buffer's tile was left before the last barrier
            if (it > 0) ask_rows(it + 1);
            if (it + 2 < n_tiles && wave == 0) ask_ids(it + 2);              // (its place held the ids of this tile)
        }
        const unsigned k_lds = lds0 + (it & 1) * BUF, v_lds = TIED ? k_lds : k_lds + PT_K * PT_ROW, rn_lds = rn_at + (it & 1) * IDS;
        auto tile = [&](auto nkb_tag) __attribute__((always_inline)) {
            constexpr int NKB = decltype(nkb_tag)::value;
            nvx_f32x16 st[NKB];
            {
                nvx_u32x4 kf[NKB][8];
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb) {
#pragma unroll
                    for (int ks = 0; ks < 8; ++ks)
                        kf[kb][ks] = *reinterpret_cast<pt_lds_u4*>((uintptr_t)(((k_lds + k_lane) ^ (ks << 5)) + kb * 32 * PT_ROW));
#pragma unroll
                    for (int r = 0; r < 16; ++r) st[kb][r] = 0.f;
                }
#pragma unroll
                for (int ks = 0; ks < 8; ++ks)
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb) st[kb] = pt_mfma(kf[kb][ks], qf[ks], st[kb], A{});
                __builtin_amdgcn_sched_group_barrier(0x100, 8 * NKB, 0);     // the reads, then the products
                __builtin_amdgcn_sched_group_barrier(0x008, 8 * NKB, 0);
            }
            // element r of block kb: key j0 + 32 kb + (r & 3) + 8 (r >> 2) + 4 half
            if (TIED) {
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                    for (int r4 = 0; r4 < 4; ++r4) {
                        const nvx_f32x4 rn = *reinterpret_cast<pt_lds_f4*>((uintptr_t)(rn_lds + 4 * (32 * kb + 8 * r4 + 4 * half)));
#pragma unroll
                        for (int r = 0; r < 4; ++r) st[kb][4 * r4 + r] *= rn[r];
                    }
            }
            if (a.cap > 0.f) {
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        st[kb][r] = k_cap - 2.0f * k_cap * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(st[kb][r] * k_lin) + 1.0f);
            } else {
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                    for (int r = 0; r < 16; ++r) st[kb][r] *= k_lin;
            }
            const float far0 = (float)(pos - j0 - 4 * half);                 // distance of the query to its first key
            if (a.r1) {
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        st[kb][r] -= pen_a * __builtin_amdgcn_logf(1.0f + pen_b * (far0 - (float)(32 * kb + (r & 3) + 8 * (r >> 2))));
            }
            if (a.slopes) {
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                    for (int r = 0; r < 16; ++r) st[kb][r] -= slope2 * (far0 - (float)(32 * kb + (r & 3) + 8 * (r >> 2)));
            }
            // most tiles: every query of the wave sees every key
            const bool full = j0 + 32 * NKB - 1 <= q_lo && (j0 >= first_seen(q_hi, a.window, a.chunk) || j0 + 32 * NKB <= a.keep);
            if (!full) {
                asm volatile("" : : : "memory");                             // (keeps the branch)
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int j = j0 + 32 * kb + (r & 3) + 8 * (r >> 2) + 4 * half;
                        st[kb][r] = j <= pos && (j >= my_lo || j < a.keep) ? st[kb][r] : -INFINITY;
                    }
            }
            float mxb[NKB];
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb) {
                mxb[kb] = st[kb][0];
#pragma unroll
                for (int r = 1; r < 16; ++r) mxb[kb] = fmaxf(mxb[kb], st[kb][r]);
            }
            float mx = NKB == 2 ? fmaxf(mxb[0], mxb[NKB - 1]) : mxb[0];
            mx = fmaxf(mx, xor32(mx));
            const float m_new = fmaxf(m_run, mx), m_ref = m_new == -INFINITY ? 0.f : m_new;
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_ref);
            m_run = m_new;
            l_run *= alpha;
            if (!__all(alpha == 1.0f)) {
#pragma unroll
                for (int d = 0; d < 4; ++d)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o_acc[d][r] *= alpha;
            }
            // 16 keys at a time: the transpose read hands a lane keys 8 (j >> 2) + 4 half + (j & 3) of them, the order of its weights
            constexpr int NG = 2 * NKB;
            typedef __attribute__((ext_vector_type(8))) short s16x8;
            s16x8 vf[NG][4];
            auto read_group = [&](int g) {
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const unsigned at = ((v_lds + v_lane) ^ (d << 6)) + g * 16 * PT_ROW;
                    const pt_s16x4 va = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<pt_lds_s16x4*>((uintptr_t)at));
                    const pt_s16x4 vb = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<pt_lds_s16x4*>((uintptr_t)((at ^ 32u) + 8 * PT_ROW)));
                    vf[g][d] = s16x8{va[0], va[1], va[2], va[3], vb[0], vb[1], vb[2], vb[3]};
                }
            };
            nvx_u32x4 p_hi[NG], p_lo[NG];
            auto weights = [&](int g) {
                const int kb = g >> 1, s2 = g & 1;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float p0 = __builtin_amdgcn_exp2f(st[kb][8 * s2 + 2 * j] - m_ref), p1 = __builtin_amdgcn_exp2f(st[kb][8 * s2 + 2 * j + 1] - m_ref);
                    l_run += p0 + p1;
                    const A h0 = (A)p0, h1 = (A)p1;
                    p_hi[g][j] = cap_pack2<A>((float)h0, (float)h1);
                    p_lo[g][j] = cap_pack2<A>(p0 - (float)h0, p1 - (float)h1);
                }
            };
            read_group(0);
            read_group(1);
            __builtin_amdgcn_sched_barrier(0);
            weights(0);
            __builtin_amdgcn_sched_barrier(0);
            // the products of a group run while the vector ALU makes the weights of the next
#pragma unroll
            for (int g = 0; g < NG; ++g) {
#pragma unroll
                for (int d = 0; d < 4; ++d) o_acc[d] = pt_mfma(__builtin_bit_cast(nvx_u32x4, vf[g][d]), p_hi[g], o_acc[d], A{});
#pragma unroll
                for (int d = 0; d < 4; ++d) o_acc[d] = pt_mfma(__builtin_bit_cast(nvx_u32x4, vf[g][d]), p_lo[g], o_acc[d], A{});
                if (g + 1 < NG) weights(g + 1);
                if (g + 2 < NG) read_group(g + 2);
                if (g + 1 < NG) {
#pragma unroll
                    for (int d = 0; d < 8; ++d) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x402, 6, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        const bool seen = wave_on && j0 < w_hi && (j0 + PT_K > w_lo || j0 < a.keep);       // some query of this wave sees some key of the tile
        if (seen && j0 + 32 < w_hi) tile(std::integral_constant<int, 2>{});
        else if (seen) tile(std::integral_constant<int, 1>{});
        pt_wait();
        __syncthreads();
    }
    // ---- the read-out: a lane holds dims 32 d + 8 r4 + 4 half + r of its query; a wave's 32 rows turn around in LDS as float32
    constexpr int OR = 132;                                                  // floats of a row there
    float* so = reinterpret_cast<float*>(smem) + wave * 32 * OR;
    if (!wave_on) return;                                                    // (no barrier follows; a wave reads back what it wrote itself)
    float l_tot = l_run + xor32(l_run);
    if (a.sink) {                                                            // one more term of the sum, no value: the maximum may move to it
        const float s2 = sink_score * LOG2E, m_new = fmaxf(m_run, s2), alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        l_tot = l_tot * alpha + __builtin_amdgcn_exp2f(s2 - m_new);
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) o_acc[d][r] *= alpha;
    }
    const float inv = a.out_mul / l_tot;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const nvx_f32x4 v = {o_acc[d][4 * r4] * inv, o_acc[d][4 * r4 + 1] * inv, o_acc[d][4 * r4 + 2] * inv, o_acc[d][4 * r4 + 3] * inv};
            *reinterpret_cast<nvx_f32x4*>(so + l32 * OR + d * 32 + 8 * r4 + 4 * half) = v;
        }
    typedef A vec8 __attribute__((ext_vector_type(8)));
    const int piece = lane & 15;
#pragma unroll
    for (int i = 0; i < 8; ++i) {                                            // four rows at a time, 16 lanes a row, eight columns a lane
        const int r = 4 * i + (lane >> 4);
        if (pb * 32 + r >= rows_here) continue;
        const int64_t tok = (int64_t)q0 + qs + pb * 32 + r;
        float o[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) o[k] = so[r * OR + piece * 8 + k];
        if (a.vcs) {                                                         // the pairs turned back by the query's angles
            const float* cs = a.vcs + tok * 128, *sn = cs + 64;
            if (a.v_inter) {
#pragma unroll
                for (int k = 0; k < 8; k += 2) {
                    const float c = cs[piece * 4 + k / 2], s = sn[piece * 4 + k / 2], u = o[k], v = o[k + 1];
                    o[k] = u * c + v * s;
                    o[k + 1] = v * c - u * s;
                }
            } else {
                const int m0 = (piece & 7) * 8;
                const float sign = piece < 8 ? 1.0f : -1.0f;                 // (u, v) -> (u c + v s, v c - u s)
#pragma unroll
                for (int k = 0; k < 8; ++k) o[k] = o[k] * cs[m0 + k] + sign * so[r * OR + (piece ^ 8) * 8 + k] * sn[m0 + k];
            }
        }
        if (a.gate && a.gate_one) {
            const float g = sigmoid_f((float)((const A*)a.gate)[tok * a.gate_stride + hd]);
#pragma unroll
            for (int k = 0; k < 8; ++k) o[k] *= g;
        } else if (a.gate) {
            const vec8 g = *reinterpret_cast<const vec8*>((const A*)a.gate + tok * a.gate_stride + (int64_t)hd * 128 + piece * 8);
#pragma unroll
            for (int k = 0; k < 8; ++k) o[k] *= sigmoid_f((float)g[k]);
        }
        vec8 w;
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = (A)o[k];
        *reinterpret_cast<vec8*>((A*)a.out + tok * a.out_stride + (int64_t)hd * 128 + piece * 8) = w;
    }
}

}  // namespace NVX_NS

using namespace NVX_NS;

int nvx_softcap_attn_rows32(const CapAttnArgs& a, int fmt, int64_t n_tok, hipStream_t st) {
    const int per_kv = a.heads / a.kv_heads, g = per_kv % 4 == 0 ? 4 : per_kv % 2 == 0 ? 2 : 1, qpos = 128 / g;
    const dim3 grid((unsigned)(a.kv_heads * (per_kv / g)), (unsigned)((n_tok + qpos - 1) / qpos + a.n_seq));
    NVX_REQUIRE(grid.y <= 65535, NVX_EINVAL, "nvx_softcap_attn: too many tokens or sequences in one step");
    const bool tied = a.k_rn != nullptr;
    // two tiles, ids and key norms; at the end 32 rows of 132 floats a wave
    const size_t loop = 2 * (tied ? 1 : 2) * PT_K * PT_ROW + 4 * PT_K * 4, end = 4 * 32 * 132 * 4, lds = loop > end ? loop : end;
#define NVX_ROWS32(A_, GG, TT)                                                                                                              \
    do {                                                                                                                                     \
        static const hipError_t attr = hipFuncSetAttribute((const void*)softcap_attn_rows32_kernel<A_, GG, TT>,                               \
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);                            \
        NVX_REQUIRE(attr == hipSuccess, NVX_ELAUNCH, "nvx_softcap_attn: cannot reserve LDS");                                                 \
        hipLaunchKernelGGL((softcap_attn_rows32_kernel<A_, GG, TT>), grid, dim3(256), lds, st, a);                                            \
    } while (0)
#define NVX_ROWS32_G(A_)                                                                  \
    do {                                                                                  \
        if (g == 4) { if (tied) NVX_ROWS32(A_, 4, true); else NVX_ROWS32(A_, 4, false); } \
        else if (g == 2) { if (tied) NVX_ROWS32(A_, 2, true); else NVX_ROWS32(A_, 2, false); } \
        else { if (tied) NVX_ROWS32(A_, 1, true); else NVX_ROWS32(A_, 1, false); }        \
    } while (0)
    if (fmt == 0) NVX_ROWS32_G(__bf16);
    else NVX_ROWS32_G(_Float16);
#undef NVX_ROWS32_G
#undef NVX_ROWS32
    return nvx_check_launch("nvx_softcap_attn");
}
