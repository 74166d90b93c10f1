// Paged prefill attention for gfx950: causal, variable length, page size 1, MFMA for QK^T and PV.
//
// Work unit = (sequence, block of query positions, kv head).  A workgroup holds, per wave, 32 query
// rows of one query head in registers (B operand of K.Q^T); the G query heads that share a kv head
// sit in different waves of the same workgroup, so every gathered K/V tile is used G times.
//
// Per 64-key tile:
//   gather   K and V rows (256 B each, located through the block table) global -> VGPR -> LDS,
//            issued one tile ahead so the HBM latency hides under the MFMAs of the current tile;
//            K rows are XOR-swizzled by (key & 15) for conflict-free ds_read_b128, V rows by
//            (key & 3) << 2 for conflict-free ds_read_b64_tr_b16;
//   S^T    = K . Q^T      v_mfma_f32_32x32x16_bf16, keys on the MFMA rows, queries on the lanes,
//            so a query's scores live in ONE lane pair: softmax needs no LDS and one lane swap;
//   P^T    = exp2(S^T - m) in fp32, rounded to bf16 in registers: the accumulator tile is already
//            the B operand of the next MFMA (k order permuted, matched by the V fragment reads);
//   O^T   += V^T . P^T    V^T fragments by the LDS transpose read; O^T keeps queries on the lanes,
//            so the online-softmax rescale is a per-lane scalar multiply.
#include "nvx_dev.h"

#include <type_traits>

namespace NVX_NS {


#define PF_KVBLK 64
#define PF_RING 4               // tiles of a workgroup with waves that only fetch: one read for values, the next for keys, one landing, one asked for
#define PF_SORTED 64             // sequences (a lane each) whose blocks are found without a plan
#define PF_IDS (2 * PF_RING)    // tiles whose slot ids such a wave keeps
#define PF_SHORT 4              // tiles up to which such a workgroup makes them one after the other
#define PF_LOG2E 1.4426950408889634f

typedef __attribute__((ext_vector_type(4))) short pf_s16x4;
typedef __attribute__((address_space(3))) pf_s16x4 pf_lds_s16x4;

// plan_ws (int32): three prefix tables, for 32, 64 and 128 query positions per workgroup:
//   table t at ws + t*(batch+2): [0] = total blocks, [1 + b] = first block of sequence b, [1 + batch] = total
#ifndef NVX_F16   // independent of the 16-bit format: defined by the bfloat16 build only
extern "C" int64_t nvx_prefill_plan_ws_ints(int64_t batch) { return 3 * (batch + 2); }
extern "C" int64_t nvx_internal_prefill_planless(void) { return PF_SORTED; }      // up to so many sequences nvx_paged_prefill reads no plan

__global__ __launch_bounds__(1024) void prefill_plan_kernel(const int32_t* __restrict__ qo_indptr, int batch,
                                                            int32_t* __restrict__ ws) {
    __shared__ int scan[1024];
    __shared__ int carry;
    const int tid = threadIdx.x;
    for (int t = 0; t < 3; ++t) {
        const int qpos = 32 << t;
        int32_t* tab = ws + t * (batch + 2);
        if (tid == 0) carry = 0;
        __syncthreads();
        for (int base = 0; base < batch; base += 1024) {
            const int b = base + tid;
            int nb = 0;
            if (b < batch) { const int lq = qo_indptr[b + 1] - qo_indptr[b]; nb = lq > 0 ? (lq + qpos - 1) / qpos : 0; }
            scan[tid] = nb;
            __syncthreads();
            for (int off = 1; off < 1024; off <<= 1) {
                const int v = tid >= off ? scan[tid - off] : 0;
                __syncthreads();
                scan[tid] += v;
                __syncthreads();
            }
            if (b < batch) tab[1 + b] = carry + scan[tid] - nb;
            __syncthreads();
            if (tid == 1023) carry += scan[1023];
            __syncthreads();
        }
        if (tid == 0) { tab[0] = carry; tab[1 + batch] = carry; }
        __syncthreads();
    }
}

extern "C" int nvx_prefill_plan(const int32_t* qo_indptr, int64_t batch, int32_t* plan_ws, int64_t plan_ws_ints,
                                nvx_stream_t stream) {
    NVX_REQUIRE(batch > 0, NVX_EINVAL, "nvx_prefill_plan: bad size");
    NVX_REQUIRE(qo_indptr && plan_ws, NVX_EINVAL, "nvx_prefill_plan: null pointer");
    NVX_REQUIRE(plan_ws_ints >= nvx_prefill_plan_ws_ints(batch), NVX_ENOSPACE, "nvx_prefill_plan: workspace too small");
    hipLaunchKernelGGL(prefill_plan_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, qo_indptr, (int)batch, plan_ws);
    return nvx_check_launch("nvx_prefill_plan");
}

#endif
// Slot ids of a tile (64 keys) travel block table -> LDS one tile before the rows they name, as ONE
// 256-byte copy issued by wave 0 (lane l fetches the id of key l).  No thread holds ids that are still
// in flight: a load issued from inline assembly hands the compiler a register whose value arrives
// later, and nothing stops the register allocator from copying that register before then (seen as rare
// wrong rows); a load the compiler knows of makes it wait for the row copies as well.
__device__ __forceinline__ void pf_dma4(const int32_t* g, unsigned lds_addr) {
    const unsigned uni = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_addr);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(g), "s"(uni) : "memory");
}
// by wave 0: ids of tile `tile` of a sequence (slot list seq_slots, lkv keys; rows past the end repeat the
// last key and are masked later) into the 64-int LDS array at `dst`
__device__ __forceinline__ void pf_fetch_slot_ids(const int32_t* __restrict__ seq_slots, int tile, int lkv, int lane, unsigned dst) {
    pf_dma4(seq_slots + min(tile * PF_KVBLK + lane, lkv - 1), dst);
}
// every vector-memory operation of this wave has completed, the copies into LDS included (the compiler
// does not know of those)
__device__ __forceinline__ void pf_wait_copies() { asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); }
// One row pair (K and V, 256 B each, 16 lanes per row) straight from the pool into LDS, no register
// staging: a wave instruction writes 64 consecutive 16-byte slots (4 rows) starting at a wave-uniform
// LDS address, so the swizzle is applied on the global side: the lane that fills position `pos` of row r
// fetches piece pos ^ swz(r).
// The copy is issued from inline assembly: through the compiler's builtin every later LDS read is held
// back until the copy has landed (the compiler cannot tell the two buffers apart), which puts the whole
// HBM latency in front of every tile.  The waits are therefore explicit: pf_wait_copies() before the
// barrier that publishes a tile.
__device__ __forceinline__ void pf_dma16(const unsigned char* g, unsigned lds_addr) {
    // lds_addr is wave-uniform by construction; the explicit broadcast puts it in a scalar register even
    // where the compiler cannot prove that.  m0 has no other user in this kernel (the toolchain refuses m0 in a clobber list: it is a reserved register).
    const unsigned uni = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_addr);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "s"(uni) : "memory");
}
// LDS reads by 32-bit LDS address (address arithmetic with XOR would hide the address space from the
// compiler if it were done on generic pointers)
typedef __attribute__((address_space(3))) const nvx_u32x4 pf_lds_u4;
__device__ __forceinline__ nvx_u32x4 pf_lds_read16(unsigned addr) { return *reinterpret_cast<pf_lds_u4*>((uintptr_t)addr); }
__device__ __forceinline__ pf_s16x4 pf_lds_read_tr(unsigned addr) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<pf_lds_s16x4*>((uintptr_t)addr));
}
__device__ __forceinline__ unsigned pf_lds_addr(const unsigned char* p) {
    return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)p;
}
// kbase / vbase already include the head and this lane's (swizzled) piece; unsigned 32-bit slot
// arithmetic keeps an address at one compare, one select and one 64-bit multiply-add
__device__ __forceinline__ void pf_gather_one(int slot_id, unsigned n_slots, const unsigned char* __restrict__ kbase,
                                              const unsigned char* __restrict__ vbase, unsigned row_bytes,
                                              unsigned k_dst, unsigned v_dst) {
    unsigned slot = (unsigned)slot_id;   // -1 -> 0xffffffff: out of range
    slot = slot < n_slots ? slot : 0u;
    const unsigned long long off = (unsigned long long)slot * row_bytes;
    pf_dma16(kbase + off, k_dst);
    pf_dma16(vbase + off, v_dst);
}
// ids: LDS address of the tile's 64 slot ids; k_dst / v_dst: start of this WAVE's four rows of pass 0 in
// the tile buffer (wave-uniform)
typedef __attribute__((address_space(3))) const int pf_lds_i32;
template <int PASSES, int KEYS_PER_PASS>
__device__ __forceinline__ void pf_gather(unsigned ids, int krow0, unsigned n_slots, const unsigned char* __restrict__ kbase,
                                          const unsigned char* __restrict__ vbase, unsigned row_bytes,
                                          unsigned k_dst, unsigned v_dst) {
    constexpr int STEP = KEYS_PER_PASS * 256;
    int id[PASSES];
#pragma unroll
    for (int p = 0; p < PASSES; ++p) id[p] = *reinterpret_cast<pf_lds_i32*>((uintptr_t)(ids + 4 * (krow0 + p * KEYS_PER_PASS)));
#pragma unroll
    for (int p = 0; p < PASSES; ++p) pf_gather_one(id[p], n_slots, kbase, vbase, row_bytes, k_dst + p * STEP, v_dst + p * STEP);
}

#if defined(PF_STAMPS) && !defined(NVX_F16)
// Build-time instrumentation (tools/build_variant.sh ... "-DPF_STAMPS"): shader-clock stamps of waves 0 and 3 of the
// workgroups of blocks 8 and 9 (kv head 0; blocks of a sequence are taken last first, so these are query blocks 119 and
// 118 of a 8 192-token sequence) at eight points of tiles 16..47, read back with nvx_debug_pf_stamps.
// Never in the shipped library.
__device__ unsigned long long pf_stamps[2 * 2 * 32 * 8];
extern "C" int nvx_debug_pf_stamps(unsigned long long* host) { return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(pf_stamps), sizeof(pf_stamps)); }
#define PF_STAMP(k) do { if (stamp_on && tile >= 16 && tile < 48 && lane == 0) \
    pf_stamps[(((stamp_blk - 8) * 2 + (wave ? 1 : 0)) * 32 + (tile - 16)) * 8 + (k)] = __builtin_readcyclecounter(); } while (0)
#else
#define PF_STAMP(k) do { } while (0)
#endif

// ---------------------------------------------------------------------------------------------
// Blocks of up to PF_SORTED sequences, longest first over all of them: sequence b has one block at each of the levels (its first query's position over
// QPOS) from its cached tokens on.  In the order of the sequences a launch of two workgroups a CU ended on whatever came last: 32 prompts of 100 to 1024 tokens, 2088
// workgroups of 15 us in the mean, 512 at a time, took 82 us.  Many short blocks (more than PF_SORT_BLOCKS, none that sees PF_SORT_KEYS) stay in the order of the
// sequences, whose neighbours share their keys in an XCD's L2.  No plan is read (two trips to memory less ahead of the first keys, and no launch of the plan).  Qwen3-0.6B, us a step by
// the plan, in order of length throughout, and by this rule (runs of one differ by 0.1-0.3 %): 8 prompts of 200-900 tokens 5590 / 5532 / 5537, 32 of 100-1024 22513 / 22240 / 22237 and
// 24184 / 24018 / 24009, 64 of 20-400 15105 / 15116 / 15060, 20 of 100-400 behind 30-1000 cached ones 8310 / 8200 / 8204, 9 of 100-400 behind 900-3000 6420 / 5834 / 5796.  One
// sequence has nothing to sort: 459 tokens by the plan, sorted, and without either 2006 / 2018 / 1995.
#define PF_SORT_BLOCKS 128
#define PF_SORT_KEYS 704
struct PfBlock { int qb, q0, lq, kv0, lkv; };       // qb < 0: there is none
__device__ __forceinline__ int pf_wave_sum(int v) {
    float f = __builtin_bit_cast(float, v);
    auto add = [&](float o) { f = __builtin_bit_cast(float, __builtin_bit_cast(int, f) + __builtin_bit_cast(int, o)); };
    add(dpp_move<0xB1>(f));
    add(dpp_move<0x4E>(f));
    add(dpp_move<0x141>(f));
    add(dpp_move<0x140>(f));
    add(xor16(f));
    add(xor32(f));
    return __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, f));
}
template <int QPOS>
__device__ __forceinline__ PfBlock pf_block_of(const int32_t* __restrict__ qo_indptr, const int32_t* __restrict__ kv_indptr, int batch, int gblk, int lane) {
    if (batch == 1) {                                // nothing to look for: last blocks first
        const int a = qo_indptr[0], n = qo_indptr[1] - a, k = kv_indptr[0], blocks = n > 0 ? (n + QPOS - 1) / QPOS : 0;
        return PfBlock{gblk < blocks ? blocks - 1 - gblk : -1, a, n, k, kv_indptr[1] - k};
    }
    int q0 = 0, q1 = 0, k0 = 0, k1 = 0;
    if (lane < batch) { q0 = qo_indptr[lane]; q1 = qo_indptr[lane + 1]; k0 = kv_indptr[lane]; k1 = kv_indptr[lane + 1]; }
    const int lq = q1 - q0, lkv = k1 - k0, nb = lq > 0 ? (lq + QPOS - 1) / QPOS : 0, base = lkv > lq ? (lkv - lq) / QPOS : 0, end = nb ? base + nb : 0;
    PfBlock w = {-1, 0, 0, 0, 0};
    const int total = pf_wave_sum(nb);
    if (gblk >= total) return w;
    auto take = [&](int b, int qb) {
        w.qb = qb;
        w.q0 = __builtin_amdgcn_readlane(q0, b);
        w.lq = __builtin_amdgcn_readlane(lq, b);
        w.kv0 = __builtin_amdgcn_readlane(k0, b);
        w.lkv = __builtin_amdgcn_readlane(lkv, b);
    };
    if (total > PF_SORT_BLOCKS && !__any(end * QPOS >= PF_SORT_KEYS)) {
        int upto = nb;
#pragma unroll
        for (int s = 1; s < 64; s <<= 1) { const int o = __shfl_up(upto, s, 64); if (lane >= s) upto += o; }
        const int b = __popcll(__ballot(upto <= gblk));
        take(b, __builtin_amdgcn_readlane(upto, b) - 1 - gblk);
        return w;
    }
    auto from_level = [&](int level) { return pf_wave_sum(min(max(end - level, 0), nb)); };
    int lo = 0, hi = 1;                              // the highest level with more than gblk blocks from it on
    while (__any(end > hi)) hi *= 2;
    while (hi - lo > 1) {
        const int mid = (lo + hi) / 2;
        if (from_level(mid) > gblk) lo = mid;
        else hi = mid;
    }
    const int nth = gblk - from_level(lo + 1);       // of the sequences that have a block of this level (a sum over the wave: not behind &&)
    const bool has = nb && base <= lo && lo < end;
    const unsigned long long there = __ballot(has);
    const int rank = __popcll(there & ((1ull << lane) - 1)), b = __ffsll((long long)__ballot(has && rank == nth)) - 1;
    take(b, lo - __builtin_amdgcn_readlane(base, b));
    return w;
}

// LOADERS > 0: that many more waves fetch the tiles, PF_RING of them in LDS, and the others only compute.  For launches that leave a CU one workgroup or little
// more: there nothing runs beside a workgroup's own chain of tiles, of whose 3450 clocks a tile the copies' addresses and issue are 600 and the wait for them 340.  With two
// workgroups a CU either hides the other's and the registers of eight more waves would not fit.  The sums are the same, bit for bit.
template <int G, int NWAVES, int LOADERS>
__global__ __launch_bounds__((NWAVES + LOADERS) * 64, LOADERS ? 1 : 2) void paged_prefill_kernel(
    const uint16_t* __restrict__ q, int64_t q_stride, const uint16_t* __restrict__ k_cache,
    const uint16_t* __restrict__ v_cache, int64_t n_slots, const int32_t* __restrict__ qo_indptr,
    const int32_t* __restrict__ kv_indptr, const int32_t* __restrict__ kv_indices, const int32_t* __restrict__ plan,
    uint16_t* __restrict__ out, int batch, int hkv, float scale_log2) {
    constexpr int NT = (NWAVES + LOADERS) * 64;
    constexpr int POSB = NWAVES / G;          // 32-row position blocks per workgroup
    constexpr int QPOS = 32 * POSB;           // query positions per workgroup
    constexpr int TAB = QPOS == 32 ? 0 : (QPOS == 64 ? 1 : 2);
    constexpr int KEYS_PER_PASS = (LOADERS ? LOADERS : NWAVES) * 4;    // 16 lanes move one 256-byte row
    constexpr int PASSES = PF_KVBLK / KEYS_PER_PASS;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    // two tile buffers of [K: 64 keys x 256 B, pieces swizzled by key & 15][V: same, swizzled by (key & 3) << 2],
    // two arrays of 64 slot ids, the counters of the owner lookup
    constexpr int BUF_BYTES = 2 * PF_KVBLK * 256;
    constexpr int IDS_BYTES = 4 * PF_KVBLK;

    const int tid = threadIdx.x, wave = LOADERS ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid >> 6, lane = tid & 63;
    const int half = lane >> 5, l32 = lane & 31;
    const int unit = blockIdx.x;
    const int gblk = unit / hkv, head = unit % hkv;
    // (the counters sit behind the tile buffers: the fragment addressing XORs address bits and needs the
    // buffers at a 256-byte boundary, which a static LDS array in front of them would break)
    constexpr int RING = LOADERS ? PF_RING : 2, ID_TILES = LOADERS ? LOADERS * PF_IDS : 2;
    int qb, q0, lq, kv0, lkv;
    if (batch <= PF_SORTED) {
        // Every wave finds the block for itself, in one trip to memory: of all sequences' blocks the one that sees the gblk-th most keys.
        const PfBlock w = pf_block_of<QPOS>(qo_indptr, kv_indptr, batch, gblk, lane);
        if (w.qb < 0) return;
        qb = w.qb; q0 = w.q0; lq = w.lq; kv0 = w.kv0; lkv = w.lkv;
    } else {
        const int32_t* tab = plan + TAB * (batch + 2);
        if (gblk >= tab[0]) return;
        // Sequence that owns query block gblk: the last b with tab[1 + b] <= gblk.  The table is
        // non-decreasing, so b + 1 is the number of entries <= gblk: every thread tests some entries and the
        // workgroup adds up.  (A binary search is log2(batch) dependent loads, several microseconds in front
        // of every workgroup's first tile; this is one.)
        int* owner_count = reinterpret_cast<int*>(smem + RING * BUF_BYTES + ID_TILES * IDS_BYTES);
        int below = 0;
        for (int i = tid; i < batch; i += NT) below += tab[1 + i] <= gblk ? 1 : 0;
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) below += __shfl_xor(below, m, 64);
        if (lane == 0) owner_count[wave] = below;
        __syncthreads();
        int b = -1;
#pragma unroll
        for (int w = 0; w < NWAVES + LOADERS; ++w) b += owner_count[w];
        b = __builtin_amdgcn_readfirstlane(b < 0 ? 0 : b);
        // blocks of a sequence are taken last first: the last query block sees the most keys, and the launch should end
        // on short blocks, not on the longest ones
        qb = tab[2 + b] - 1 - gblk;
        q0 = qo_indptr[b]; lq = qo_indptr[b + 1] - q0;
        kv0 = kv_indptr[b]; lkv = kv_indptr[b + 1] - kv0;
    }
    const int offset = lkv - lq;              // query i sees keys 0 .. i + offset
    const int g = wave % G, pb = wave / G;
    const int qi = qb * QPOS + pb * 32 + l32;  // this lane's query (position within the new tokens)
    const bool q_ok = qi < lq;
    const int hq_total = hkv * G;
    const int hq = head * G + g;
    int kmax = qb * QPOS + QPOS + offset;       // keys visible to the workgroup's last query
    kmax = kmax > lkv ? lkv : kmax;
    const int wave_last_key = qb * QPOS + pb * 32 + 31 + offset;  // last key any query of this wave sees
    const int wave_first_vis = qb * QPOS + pb * 32 + offset;      // last key the wave's FIRST query sees
    const int n_tiles = (max(kmax, 0) + PF_KVBLK - 1) / PF_KVBLK;

    if constexpr (LOADERS > 0) {
        if (wave >= NWAVES) {
            // A loader wave has the same keys of every tile, and every tile's ids in LDS of its own, PF_RING tiles before their rows (operations complete
            // in order, so the wait for a tile's rows is a wait for the ids of the rows that are asked for next).
            const int me = wave - NWAVES, pos = lane & 15, krow0 = me * 4 + (lane >> 4);
            const int32_t* seq_slots = kv_indices + kv0;
            const unsigned char* kg = reinterpret_cast<const unsigned char*>(k_cache) + head * 256 + ((pos ^ (krow0 & 15)) << 4);
            const unsigned char* vg = reinterpret_cast<const unsigned char*>(v_cache) + head * 256 + ((pos ^ ((krow0 & 3) << 2)) << 4);
            const unsigned n_slots_u = n_slots > 0xffffffffll ? 0xffffffffu : (unsigned)n_slots;
            const unsigned lds0 = pf_lds_addr(smem), rows = (unsigned)__builtin_amdgcn_readfirstlane(me * 4 * 256);
            const unsigned ids = lds0 + (unsigned)__builtin_amdgcn_readfirstlane(RING * BUF_BYTES + me * PF_IDS * IDS_BYTES);
            auto fetch_ids = [&](int t) { pf_fetch_slot_ids(seq_slots, t, lkv, lane, ids + (t % PF_IDS) * IDS_BYTES); };
            // where a tile's rows lie is found a turn before they are asked for: behind a barrier nothing is in front of the copies
            unsigned long long from[PASSES];
            auto find_rows = [&](int t) __attribute__((always_inline)) {
                const unsigned at = ids + (t % PF_IDS) * IDS_BYTES;
#pragma unroll
                for (int p = 0; p < PASSES; ++p) {
                    unsigned slot = (unsigned)*reinterpret_cast<pf_lds_i32*>((uintptr_t)(at + 4 * (krow0 + p * KEYS_PER_PASS)));
                    slot = slot < n_slots_u ? slot : 0u;
                    from[p] = (unsigned long long)slot * ((unsigned)hkv * 256u);
                }
            };
            auto fetch_rows = [&](int t) __attribute__((always_inline)) {
                const unsigned at = lds0 + (unsigned)(t % RING) * BUF_BYTES + rows;
#pragma unroll
                for (int p = 0; p < PASSES; ++p) {
                    pf_dma16(kg + from[p], at + p * (KEYS_PER_PASS * 256));
                    pf_dma16(vg + from[p], at + PF_KVBLK * 256 + p * (KEYS_PER_PASS * 256));
                }
            };
            for (int t = 0; t < n_tiles && t < 2 * RING - 1; ++t) fetch_ids(t);
            pf_wait_copies();
            // Few tiles: a turn that makes the scores of the tile behind it has little to hide there, waits for a second tile ahead of the first, and makes scores of keys that nobody sees.  us a launch, the
            // loop with such waves alone (before there were turns), turns alone, and this: 20 tokens 4.31, 4.82, 4.23; 100 5.82, 6.12, 5.65; 200 7.48, 7.75, 7.12; 459 11.9, 11.7, 11.2 (between
            // products 12.6, 12.5, 11.1); 1000 21.4, 19.9, 19.2; four of 100 6.50, 6.86, 6.31.  Turns from the third tile on: 200 tokens 7.46, four of 200 8.43 instead of 8.09; from the sixth: the same as from the fifth.
            if (n_tiles <= PF_SHORT) {
                // tile t's turn begins when tile t has landed; two are on their way, and no ids are left to ask for
                static_assert(PF_SHORT < 2 * PF_RING, "ids of a short run");
                for (int t = -2; t < n_tiles; ++t) {
                    if (t + 2 < n_tiles) {
                        find_rows(t + 2);
                        fetch_rows(t + 2);                                         // (to where tile t - 2 was)
                    }
                    if (t == -2) continue;
                    if (t + 2 < n_tiles) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * PASSES) : "memory");
                    else pf_wait_copies();
                    __syncthreads();
                }
                return;
            }
            for (int t = 0; t < RING - 1; ++t) {
                find_rows(t);
                fetch_rows(t);
            }
            static_assert(RING == 4 && PF_SHORT >= RING - 2, "what may be on its way at a barrier: the rows of one tile");
            find_rows(RING - 1);                                                   // (whatever lies there if there is no such tile: not used)
            // tile t's turn begins when tile t + 1 has landed
            asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * PASSES) : "memory");
            __syncthreads();
            for (int t = 0; t < n_tiles; ++t) {
                const bool more_rows = t + RING - 1 < n_tiles, more_ids = t + 2 * RING - 1 < n_tiles;
                if (more_rows) fetch_rows(t + RING - 1);                           // (to where tile t - 1 was)
                if (more_ids) fetch_ids(t + 2 * RING - 1);
                find_rows(t + RING);                                               // (its ids came with tile t - 3's turn)
                // all but what this turn asked for: tile t + 2 has landed
                if (more_ids) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * PASSES + 1) : "memory");
                else if (more_rows) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * PASSES) : "memory");
                else pf_wait_copies();
                __syncthreads();
            }
            return;
        }
    }
    // Q^T fragments: 8 k-steps of 16 dims; lane holds dims 16*ks + 8*half .. +7 of its query row
    nvx_h16x8 qf[8];
    {
        const uint16_t* qrow = q + (int64_t)(q0 + (q_ok ? qi : 0)) * q_stride + hq * 128 + half * 8;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            uint4 t = *reinterpret_cast<const uint4*>(qrow + ks * 16);
            if (!q_ok) t = make_uint4(0, 0, 0, 0);
            qf[ks] = __builtin_bit_cast(nvx_h16x8, t);
        }
    }

    nvx_f32x16 o_acc[4];
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[d][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    static_assert(PASSES == 2 || PASSES == 4, "tile gather is written for four or eight waves");
    // Pipeline, one barrier per tile: while tile t is computed from one buffer, the rows of tile t + 1 travel
    // pool -> LDS into the other and the slot ids of tile t + 2 block table -> LDS.
    const int pos = tid & 15, krow0 = tid >> 4;
    const int32_t* seq_slots = kv_indices + kv0;
    // this lane's piece of a row: KEYS_PER_PASS is a multiple of 16, so the swizzle is the same for every pass
    const unsigned char* kg = reinterpret_cast<const unsigned char*>(k_cache) + head * 256 + ((pos ^ (krow0 & 15)) << 4);
    const unsigned char* vg = reinterpret_cast<const unsigned char*>(v_cache) + head * 256 + ((pos ^ ((krow0 & 3) << 2)) << 4);
    const unsigned row_bytes = (unsigned)hkv * 256u;
    const unsigned n_slots_u = n_slots > 0xffffffffll ? 0xffffffffu : (unsigned)n_slots;
    const unsigned wave_rows = (unsigned)__builtin_amdgcn_readfirstlane(wave * 4 * 256);
    const unsigned lds0 = pf_lds_addr(smem);
    // per-lane byte offsets of the fragment reads inside a tile buffer (see the reads below)
    const int k_lane_off = l32 * 256 + ((half ^ (l32 & 15)) << 4);
    const int v_lane_off = [&] {
        const int grp = lane >> 4, i16 = lane & 15, tq = i16 >> 2, tp = i16 & 3;
        const int row = 4 * half + tq;
        const int pc0 = 2 * (grp & 1) + (tp >> 1);
        return row * 256 + ((pc0 ^ ((row & 3) << 2)) << 4) + 8 * (tp & 1);
    }();
    unsigned ring0 = lds0, ring1 = lds0 + BUF_BYTES;                 // tile being computed, tile arriving
    unsigned ids0 = lds0 + 2 * BUF_BYTES, ids1 = ids0 + IDS_BYTES;     // slot ids of the next tile, of the one after
    if (LOADERS == 0 && n_tiles > 0) {
        if (wave == 0) {
            pf_fetch_slot_ids(seq_slots, 0, lkv, lane, ids0);
            if (n_tiles > 1) pf_fetch_slot_ids(seq_slots, 1, lkv, lane, ids1);
        }
        pf_wait_copies();
        __syncthreads();
        // the first TWO tiles travel together: a workgroup's first round trip to the pool is the one nothing
        // can hide, so it carries as much as the buffers hold
        pf_gather<PASSES, KEYS_PER_PASS>(ids0, krow0, n_slots_u, kg, vg, row_bytes, ring0 + wave_rows, ring0 + PF_KVBLK * 256 + wave_rows);
        if (n_tiles > 1)
            pf_gather<PASSES, KEYS_PER_PASS>(ids1, krow0, n_slots_u, kg, vg, row_bytes, ring1 + wave_rows, ring1 + PF_KVBLK * 256 + wave_rows);
        pf_wait_copies();
    }
    __syncthreads();
    { const unsigned t0 = ids0; ids0 = ids1; ids1 = t0; }
    bool made = false;
    if constexpr (LOADERS > 0) if (n_tiles > PF_SHORT) {
        // A turn: the sums of values of `tile` and the scores of the tile behind it.  A wave that has its SIMD to itself and makes a tile's scores, their probabilities and the sums
        // of values one after the other lets the matrix pipe wait for the vector ALU and the other way round; here every group of products has exponentials or maxima beside
        // it, and a turn begins under the last products of the one before.  All chains of sums run as in the loop below.  Alone and with its keys in the caches a turn takes 0.86 us, of which the matrix
        // pipe needs 0.43 (64 queries of 3072 keys 54.2 us before, 46.8 now; 43.6 if weights were relative to a score that later ones may exceed by 2^8, which spares most of the accumulators' multiplications
        // but rounds the largest weight, and so results: 1.00 to 1.24 of the error against 64 bits).
        typedef __attribute__((ext_vector_type(8))) short s16x8;
        const int vis = q_ok ? qi + offset : -1;                                          // last key this lane's query sees
        // 32-key blocks of a tile that hold keys some query of the wave sees (wave-uniform)
        const int tiles_u = __builtin_amdgcn_readfirstlane(n_tiles), last_u = __builtin_amdgcn_readfirstlane(wave_last_key), first_u = __builtin_amdgcn_readfirstlane(wave_first_vis);
        auto blocks_of = [&](int t) { return t >= tiles_u || t * PF_KVBLK > last_u ? 0 : t * PF_KVBLK + 32 <= last_u ? 2 : 1; };
        nvx_f32x16 st[2];                                                                 // scores of the next tile
        float ex[2][16], mx[2], alpha = 0.f;                                              // what the exponentials of the present one are taken of; the largest; what becomes of the sums so far
        nvx_u32x4 keys[8];                                                                // the next tile's first block
        // half of the columns of a tile's keys: both blocks of 32, whose products take turns (0.88 us a tile where a block's eight in a row were 0.91)
        auto read_keys = [&](nvx_u32x4 (&kf)[8], int t, int h) __attribute__((always_inline)) {
            const unsigned at = lds0 + (unsigned)(t % RING) * BUF_BYTES + k_lane_off;
#pragma unroll
            for (int i = 0; i < 8; ++i) kf[i] = pf_lds_read16((at ^ ((4 * h + (i >> 1)) << 5)) + (i & 1) * 32 * 256);
        };
        auto multiply_keys = [&](const nvx_u32x4 (&kf)[8], int h) __attribute__((always_inline)) {
            if (h == 0) {
#pragma unroll
                for (int r = 0; r < 16; ++r) st[0][r] = st[1][r] = 0.f;
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) st[i & 1] = mfma_32x32x16_h16(__builtin_bit_cast(nvx_h16x8, kf[i]), qf[4 * h + (i >> 1)], st[i & 1]);
        };
        auto mask = [&](int t) __attribute__((always_inline)) {
            if (t * PF_KVBLK + PF_KVBLK - 1 <= first_u) return;                           // wave-uniform
            const int upto = vis - t * PF_KVBLK - 4 * half;
            asm volatile("" : : : "memory");
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r) st[kb][r] = kb * 32 + (r & 3) + 8 * (r >> 2) <= upto ? st[kb][r] : -INFINITY;
        };
        auto maximum = [&](int kb) __attribute__((always_inline)) {
            mx[kb] = st[kb][0];
#pragma unroll
            for (int r = 1; r < 16; ++r) mx[kb] = fmaxf(mx[kb], st[kb][r]);
        };
        uint32_t pw[4][4];                                                                 // P^T, 16 keys a group
        auto half_group = [&](int h) __attribute__((always_inline)) {                      // four exponentials per lane
            const int gi = h >> 1, j0 = 2 * (h & 1);
#pragma unroll
            for (int j = j0; j < j0 + 2; ++j) {
                const float p0 = __builtin_amdgcn_exp2f(ex[gi >> 1][8 * (gi & 1) + 2 * j]);
                const float p1 = __builtin_amdgcn_exp2f(ex[gi >> 1][8 * (gi & 1) + 2 * j + 1]);
                l_run = h == 0 && j == 0 ? fmaf(l_run, alpha, p0 + p1) : l_run + (p0 + p1);
                pw[gi][j] = pack_h16x2(p0, p1);
            }
            asm volatile("" : "+v"(pw[gi][j0]), "+v"(pw[gi][j0 + 1]), "+v"(l_run));        // here, and not behind the next branch, where the products need them
        };
        float mref = 0.f;
        auto begin = [&]() __attribute__((always_inline)) {
            float m = fmaxf(mx[0], mx[1]);
            m = fmaxf(m, xor32(m));
            const float m_new = fmaxf(m_run, m * scale_log2);     // scale_log2 > 0
            mref = m_new == -INFINITY ? 0.f : m_new;
            alpha = __builtin_amdgcn_exp2f(m_run - mref);
            m_run = m_new;
        };
        auto exponents = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) ex[kb][r] = fmaf(st[kb][r], scale_log2, -mref);
        };
        // `tile`, begun, whose first NKB blocks are multiplied with values, and the scores of the tile behind it if NEXT (what that has beyond its last key is masked)
        auto turn = [&](auto nkb_tag, auto next_tag, int tile) __attribute__((always_inline)) {
            constexpr int NKB = decltype(nkb_tag)::value, NEXT = decltype(next_tag)::value ? 2 : 0, NGRP = 2 * NKB, STAGES = NEXT + NGRP;   // groups of 16 keys; of products
            const unsigned vfrag0 = lds0 + (unsigned)(tile % RING) * BUF_BYTES + PF_KVBLK * 256 + v_lane_off;
            nvx_u32x4 second[8];
            s16x8 vf[NGRP][4];
            auto read_group = [&](int gi) __attribute__((always_inline)) {                // V^T fragments, as below
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const unsigned pa = (vfrag0 ^ (d << 6)) + gi * 16 * 256;
                    const pf_s16x4 va = pf_lds_read_tr(pa);
                    const pf_s16x4 vb = pf_lds_read_tr(pa + 8 * 256);
                    vf[gi][d] = s16x8{va[0], va[1], va[2], va[3], vb[0], vb[1], vb[2], vb[3]};
                }
            };
            if (NEXT == 0) {
                read_group(0);
                half_group(0);
                half_group(1);
            }
#pragma unroll
            for (int i = 0; i < STAGES; ++i) {
                if (NEXT > 0 && i == NEXT) mask(tile + 1);
                if (i == NEXT && !__all(alpha == 1.0f)) {
#pragma unroll
                    for (int d = 0; d < 4; ++d)
#pragma unroll
                        for (int r = 0; r < 16; ++r) o_acc[d][r] *= alpha;
                }
                if (i == STAGES - 1) {                                                    // everything of this tile is in registers
                    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");                  // (a barrier alone does not wait for reads)
                    __syncthreads();                                                      // tile + 2 has landed, this one's place is free
                    if (NEXT > 0) read_keys(keys, tile + 2, 0);                           // (whatever lies there if there is no such tile: not used)
                }
                __builtin_amdgcn_sched_barrier(0);
                // products: a block's scores, then a group's values
                if (i < NEXT) {
                    multiply_keys(i == 0 ? keys : second, i);
                } else {
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        const uint32_t* w = pw[i - NEXT];
                        o_acc[d] = mfma_32x32x16_h16(__builtin_bit_cast(nvx_h16x8, vf[i - NEXT][d]), __builtin_bit_cast(nvx_h16x8, make_uint4(w[0], w[1], w[2], w[3])), o_acc[d]);
                    }
                }
                // reads for what comes next
                if (i + 1 < NEXT) read_keys(second, tile + 1, 1);
                else if (i + 1 < STAGES) read_group(i + 1 - NEXT);
                // beside them, dealt out by what they cost: a group's exponentials are as long as four to six of the products
                if (NEXT == 0) {
                    if (i + 1 < NGRP) {
                        half_group(2 * i + 2);
                        half_group(2 * i + 3);
                    }
                } else if (i < 2) {
                    half_group(3 * i);
                    half_group(3 * i + 1);
                    half_group(3 * i + 2);
                } else if (i == 2) {
                    half_group(6);
                    half_group(7);
                } else if (i == 3) {
                    maximum(0);
                    maximum(1);
                } else if (i == 4) {
                    begin();
                } else {
                    exponents(0);
                    exponents(1);
                }
                if (i < NEXT) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x400, 2, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                        __builtin_amdgcn_sched_group_barrier(0x400, 2, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        int tile = 0;
        if (blocks_of(0) > 0) {
            read_keys(keys, 0, 0);
            multiply_keys(keys, 0);
            read_keys(keys, 0, 1);
            multiply_keys(keys, 1);
            read_keys(keys, 1, 0);                                  // (whatever lies there if there is no such tile: not used)
            mask(0);
            maximum(0);
            maximum(1);
            begin();
            exponents(0);
            exponents(1);
            for (; blocks_of(tile + 1) > 0; ++tile) turn(std::integral_constant<int, 2>{}, std::true_type{}, tile);
            if (blocks_of(tile) == 2) turn(std::integral_constant<int, 2>{}, std::false_type{}, tile);
            else turn(std::integral_constant<int, 1>{}, std::false_type{}, tile);
            ++tile;
        }
        for (; tile < n_tiles; ++tile) __syncthreads();      // (nothing of these is visible to this wave)
        made = true;
    }
    if (!made) {
    // at the top of tile t: ids0 holds the ids of tile t + 1, ids1 is free (its ids were used a tile ago)
#ifdef PF_STAMPS
    const int stamp_blk = gblk;
    const bool stamp_on = (gblk == 8 || gblk == 9) && head == 0 && (wave == 0 || wave == 3);
#endif
    // (a branch of lanes: behind a uniform one the accumulators move between two sets of registers three times a tile, 0.2 us of it)
    int last_key = wave_last_key;
    if (LOADERS) asm volatile("" : "+v"(last_key));
    for (int tile = 0; tile < n_tiles; ++tile) {
        PF_STAMP(0);
        const unsigned k_lds = ring0;   // LDS byte addresses
        const unsigned v_lds = k_lds + PF_KVBLK * 256;
        if (LOADERS == 0 && tile + 1 < n_tiles) {   // the other buffer held tile t - 1: every wave left it before the last barrier
            if (tile > 0)           // (tile 1 came with tile 0)
                pf_gather<PASSES, KEYS_PER_PASS>(ids0, krow0, n_slots_u, kg, vg, row_bytes, ring1 + wave_rows, ring1 + PF_KVBLK * 256 + wave_rows);
            if (tile + 2 < n_tiles && wave == 0) pf_fetch_slot_ids(seq_slots, tile + 2, lkv, lane, ids1);
        }

        PF_STAMP(1);
        const int key_base = tile * PF_KVBLK;
        // One tile for this wave: NKB = 2 when both 32-key blocks hold keys some query of the wave sees, 1 when the
        // second block lies wholly beyond the causal diagonal for all of them (half the waves of a workgroup on
        // its last tile): its score and value MFMAs, exponentials and LDS reads are then not issued at all.
        auto tile_body = [&](auto nkb_tag) __attribute__((always_inline)) {
        constexpr int NKB = decltype(nkb_tag)::value;

        // ---- S^T = K . Q^T ----
        // all K fragments are requested before the first MFMA, and the 32-key blocks alternate so that no MFMA
        // waits for the one before it
        nvx_f32x16 st[NKB];
        nvx_u32x4 kf[NKB][8];
        // fragment ks of key row l32 (+32 for the second block) sits at piece (2 ks + half) ^ (key & 15): one
        // per-tile base, the k-step applied as an XOR on the address bits, the block as an immediate offset
        const unsigned kfrag0 = k_lds + k_lane_off;
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
#pragma unroll
            for (int ks = 0; ks < 8; ++ks)
                kf[kb][ks] = pf_lds_read16((kfrag0 ^ (ks << 5)) + kb * 32 * 256);
#pragma unroll
            for (int r = 0; r < 16; ++r) st[kb][r] = 0.f;
        }
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
                st[kb] = mfma_32x32x16_h16(__builtin_bit_cast(nvx_h16x8, kf[kb][ks]), qf[ks], st[kb]);
        // scheduling order for this region: the LDS reads, then the MFMAs
        __builtin_amdgcn_sched_group_barrier(0x100, 8 * NKB, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 8 * NKB, 0);
        PF_STAMP(2);
        // ---- mask, online softmax (this lane: one query, 16 of each 32-key block) ----
        // Scores stay unscaled; the scale rides on the fused multiply-add inside the exponent.  Only
        // tiles that cross the causal diagonal (or the end of the sequence) pay for the mask.
        const int vis = q_ok ? qi + offset : -1;   // last visible key index of this lane's query
        if (key_base + 32 * NKB - 1 > wave_first_vis) {   // wave-uniform
            asm volatile("" : : : "memory");   // keeps the branch: as selects on every tile the mask costs 96 VALU ops
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = key_base + kb * 32 + (r & 3) + 8 * (r >> 2) + 4 * half;
                    st[kb][r] = key <= vis ? st[kb][r] : -INFINITY;
                }
        }
        // (one chain of maxima per 32-key block: the chains are dependent instructions, and two run side by side)
        float mxb[NKB];
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
            mxb[kb] = st[kb][0];
#pragma unroll
            for (int r = 1; r < 16; ++r) mxb[kb] = fmaxf(mxb[kb], st[kb][r]);
        }
        float mx = NKB == 2 ? fmaxf(mxb[0], mxb[NKB - 1]) : mxb[0];
        mx = fmaxf(mx, xor32(mx));
        const float m_new = fmaxf(m_run, mx * scale_log2);     // scale_log2 > 0
        const float mref = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m_run - mref);
        m_run = m_new;
        if (!__all(alpha == 1.0f)) {
#pragma unroll
            for (int d = 0; d < 4; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) o_acc[d][r] *= alpha;
        }
        PF_STAMP(3);
        // ---- P^T, then O^T += V^T . P^T ----
        // V^T fragment element j of lane half h is key 16*s2 + 8*(j>>2) + 4*h + (j&3) of the 32-key block; the
        // transpose read hands lane i of a 16-lane group column i of a 4-key x 16-dim block.  The lane
        // addresses row 4 half + tq (+ 16 s2 + 32 kb, and + 8 for the second read: immediate offsets); the
        // dim block d enters the swizzled piece index as an XOR on address bits 6-7.
        // Order, fixed with scheduling barriers because the compiler otherwise sinks every LDS read to
        // just before its MFMA and waits out the LDS latency 32 times per tile: the V fragments of the
        // first two (kb, s2) groups are requested before the exponentials and land under them; each group
        // of four MFMAs is followed by the reads of the group two ahead.
        typedef __attribute__((ext_vector_type(8))) short s16x8;
        constexpr int NGRP = 2 * NKB;   // groups of 16 keys
        const unsigned vfrag0 = v_lds + v_lane_off;
        s16x8 vf[NGRP][4];
        auto read_group = [&](int grp_i) {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const unsigned pa = (vfrag0 ^ (d << 6)) + grp_i * 16 * 256;   // group = 2 kb + s2: 16 keys each
                const pf_s16x4 va = pf_lds_read_tr(pa);
                const pf_s16x4 vb = pf_lds_read_tr(pa + 8 * 256);
                vf[grp_i][d] = s16x8{va[0], va[1], va[2], va[3], vb[0], vb[1], vb[2], vb[3]};
            }
        };
        read_group(0);
        read_group(1);
        __builtin_amdgcn_sched_barrier(0);
        nvx_h16x8 pf[NGRP];
        auto probabilities = [&](int gi) {   // P^T of 16 keys: 8 exponentials per lane
            const int kb = gi >> 1, s2 = gi & 1;
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float p0 = __builtin_amdgcn_exp2f(fmaf(st[kb][8 * s2 + 2 * j], scale_log2, -mref));
                const float p1 = __builtin_amdgcn_exp2f(fmaf(st[kb][8 * s2 + 2 * j + 1], scale_log2, -mref));
                l_run = gi == 0 && j == 0 ? fmaf(l_run, alpha, p0 + p1) : l_run + (p0 + p1);
                w[j] = pack_h16x2(p0, p1);
            }
            pf[gi] = __builtin_bit_cast(nvx_h16x8, make_uint4(w[0], w[1], w[2], w[3]));
        };
        probabilities(0);
        __builtin_amdgcn_sched_barrier(0);
        PF_STAMP(4);
        // the four MFMAs of a group run on the matrix pipe while the vector ALU makes the next group's
        // probabilities: one MFMA, then a share of the exponentials, four times over
#pragma unroll
        for (int gi = 0; gi < NGRP; ++gi) {
#pragma unroll
            for (int d = 0; d < 4; ++d)
                o_acc[d] = mfma_32x32x16_h16(__builtin_bit_cast(nvx_h16x8, vf[gi][d]), pf[gi], o_acc[d]);
            if (gi + 1 < NGRP) probabilities(gi + 1);
            if (gi + 2 < NGRP) read_group(gi + 2);
            if (gi + 1 < NGRP) {
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x402, 8, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        PF_STAMP(5);
        };
        if (key_base + 32 <= last_key) tile_body(std::integral_constant<int, 2>{});        // wave-uniform
        else if (key_base <= last_key) tile_body(std::integral_constant<int, 1>{});        // else: nothing visible
        if (LOADERS == 0) pf_wait_copies();
        PF_STAMP(6);
        __syncthreads();   // tile + 1 and the ids of tile + 2 visible; this tile's buffer free
        PF_STAMP(7);
        if (LOADERS) ring0 = ring0 == lds0 + (RING - 1) * BUF_BYTES ? lds0 : ring0 + BUF_BYTES;
        else { const unsigned t0 = ring0; ring0 = ring1; ring1 = t0; }
        { const unsigned t0 = ids0; ids0 = ids1; ids1 = t0; }
    }
    }

    // ---- epilogue: O = O^T / l ----
    // A lane holds 64 of the 128 dims of ONE query row, so stores straight from registers are 64 scattered
    // 8-byte writes per instruction (a third of the kernel's time on short sequences).  Each wave instead
    // turns its 32 x 128 block around in LDS (the tile buffers are free: the loop ended with a barrier;
    // rows 272 B apart keep the 8-byte writes off each other's banks and the 16-byte reads aligned) and
    // stores whole 256-byte rows, four per instruction.
    const float l_tot = l_run + xor32(l_run);
    {
        constexpr int ROW = 272;
        const unsigned stage = lds0 + (unsigned)__builtin_amdgcn_readfirstlane(wave * 32 * ROW);
        const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
        typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
        typedef __attribute__((address_space(3))) u32x2 lds_u2;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                const int dim = d * 32 + 8 * r4 + 4 * half;
                *reinterpret_cast<lds_u2*>((uintptr_t)(stage + l32 * ROW + dim * 2)) =
                    u32x2{pack_h16x2(o_acc[d][4 * r4] * inv, o_acc[d][4 * r4 + 1] * inv),
                          pack_h16x2(o_acc[d][4 * r4 + 2] * inv, o_acc[d][4 * r4 + 3] * inv)};
            }
        // a wave's LDS operations complete in order: no barrier between its writes and its reads
        const int rq = lane >> 4, pc = lane & 15;
        const int q_first = qb * QPOS + pb * 32;   // the wave's first query position
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int row = 4 * i + rq;
            const nvx_u32x4 v = pf_lds_read16(stage + row * ROW + pc * 16);
            if (q_first + row < lq)
                *reinterpret_cast<nvx_u32x4*>(out + ((int64_t)(q0 + q_first + row) * hq_total + hq) * 128 + pc * 8) = v;
        }
    }
}

// Workgroups of so many query positions, at most
static int64_t pf_groups(int64_t positions, int64_t n_tokens, int64_t batch, int64_t hkv) { return ((n_tokens + positions - 1) / positions + batch - 1) * hkv; }
// Few workgroups: waves of their own for the copies, and where there are fewer still 32 positions of two heads as two waves, which read half as much LDS a tile.  us a launch
// with loader waves and the loop without them, 16 query heads: one sequence of 459 tokens 11.2 (32 positions) and 13.5.  Figures of turns that took 0.79 us (see there): 64 positions: 2500 tokens 43.1 and 57.3, six
// questions behind 900-3000 keys (272 workgroups) 56.7 and 74.4, twelve (560) 93.0 and 80.8, eight prompts of 100-1024 (648) 35.6 and 31.3, 32 of 20-60 (416) 7.1 and 6.5.  32 heads: 1500 tokens 29.0
// and 38.1, 2000 (504) 44.2 and 51.2, 20 of 30-100 behind 900 (488) 46.5 and 39.2, 632 70 and 67.
// Between 392 and 512 workgroups what decides is how uneven the blocks are, of which the host knows the tokens and the sequences only: one or two sequences' blocks see more and more keys, and the longest are done
// first.  us a step of Qwen3-0.6B with loader waves and without, 400 to 512 workgroups: one sequence 0.94 to 0.97 of the time (3168 tokens 6445 and 6830), also behind 700 and 2500 keys; two of one length
// 0.97 to 1.00, two of 0.4 and 1.6 times their mean 0.93 to 0.97; three or more of one length up to 1.05 (eight of 452 tokens 5324 and 5215, ten of 272 behind 400 keys 5202 and 4953; as many uneven ones 0.93 to 1.04).  Four layers
// of Qwen3-8B: one sequence 0.985 to 1.01; two 0.99 to 1.01, more 1.00 to 1.02.
static bool pf_loaders(int g, int64_t n_tokens, int64_t batch, int64_t hkv) {
    return (g == 2 || g == 4) && pf_groups(g == 2 ? 64 : 32, n_tokens, batch, hkv) <= (batch <= (g == 2 ? 2 : 1) ? 512 : 392);
}
extern "C" int NVX_ENTRY(nvx_internal_prefill_loaders)(int64_t n_tokens, int64_t batch, int n_q_heads, int n_kv_heads) { return pf_loaders(n_q_heads / n_kv_heads, n_tokens, batch, n_kv_heads); }

extern "C" int NVX_ENTRY(nvx_paged_prefill)(const void* q, int64_t q_row_stride, const void* k_cache, const void* v_cache,
                                 int64_t n_slots, const int32_t* qo_indptr, const int32_t* kv_indptr,
                                 const int32_t* kv_indices, const int32_t* plan_ws, void* out, int64_t n_tokens,
                                 int64_t batch, int n_q_heads, int n_kv_heads, float sm_scale, nvx_stream_t stream) {
    NVX_REQUIRE(batch > 0 && n_tokens >= 0 && n_q_heads > 0 && n_kv_heads > 0 && n_slots > 0, NVX_EINVAL, "nvx_paged_prefill: bad size");
    if (n_tokens == 0) return NVX_OK;
    NVX_REQUIRE(q && k_cache && v_cache && qo_indptr && kv_indptr && kv_indices && plan_ws && out, NVX_EINVAL,
                "nvx_paged_prefill: null pointer");
    NVX_REQUIRE(n_q_heads % n_kv_heads == 0, NVX_EINVAL, "nvx_paged_prefill: n_q_heads must be a multiple of n_kv_heads");
    NVX_REQUIRE(q_row_stride % 8 == 0 && q_row_stride >= (int64_t)n_q_heads * 128, NVX_EINVAL, "nvx_paged_prefill: bad q row stride");
    NVX_REQUIRE(nvx_aligned16(q) && nvx_aligned16(k_cache) && nvx_aligned16(v_cache) && nvx_aligned16(out), NVX_EINVAL,
                "nvx_paged_prefill: pointers must be 16-byte aligned");
    const int g = n_q_heads / n_kv_heads;
    const float scale_log2 = sm_scale * PF_LOG2E;
    hipStream_t st = (hipStream_t)stream;
    // two tile buffers of K and V, two tiles of slot ids, per-wave counters; at the end the same memory
    // stages the output, 32 rows of 272 B per wave
    const size_t loop_bytes = 2 * 2 * PF_KVBLK * 256 + 2 * 4 * PF_KVBLK + 64;
#define NVX_PF(GG, NW, QPOS, LD)                                                                                       \
    do {                                                                                                                \
        const size_t need = (LD) ? (size_t)PF_RING * 2 * PF_KVBLK * 256 + (size_t)(LD) * PF_IDS * 4 * PF_KVBLK + 64 : loop_bytes; \
        const size_t lds_bytes = need > (size_t)(NW) * 32 * 272 ? need : (size_t)(NW) * 32 * 272;                       \
        static const hipError_t attr = hipFuncSetAttribute((const void*)paged_prefill_kernel<GG, NW, LD>,               \
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes); \
        NVX_REQUIRE(attr == hipSuccess, NVX_ELAUNCH, "nvx_paged_prefill: cannot reserve %d KB of LDS", (int)(lds_bytes / 1024)); \
        const int64_t blocks = ((n_tokens + (QPOS) - 1) / (QPOS) + batch) * n_kv_heads;                                 \
        hipLaunchKernelGGL((paged_prefill_kernel<GG, NW, LD>), dim3((unsigned)blocks), dim3(((NW) + (LD)) * 64), lds_bytes, st, \
                           (const uint16_t*)q, q_row_stride, (const uint16_t*)k_cache, (const uint16_t*)v_cache,        \
                           n_slots, qo_indptr, kv_indptr, kv_indices, plan_ws, (uint16_t*)out, (int)batch, n_kv_heads,  \
                           scale_log2);                                                                                 \
    } while (0)
    const bool loaders = pf_loaders(g, n_tokens, batch, n_kv_heads);
    switch (g) {
        case 1: NVX_PF(1, 4, 128, 0); break;
        // two 4-wave workgroups per CU (each in its own phase of the tile loop) measured faster than one
        // 8-wave workgroup of 128 queries (0.75 vs 0.86 ms on the bench prompts); a third tile buffer (row
        // copies two tiles ahead) changed neither
        case 2:
            if (pf_groups(32, n_tokens, batch, n_kv_heads) <= 256) NVX_PF(2, 2, 32, 4);
            else if (loaders) NVX_PF(2, 4, 64, 4);
            else NVX_PF(2, 4, 64, 0);
            break;
        case 4:
            if (loaders) NVX_PF(4, 4, 32, 4);
            else NVX_PF(4, 4, 32, 0);
            break;   // 8 waves / 64 queries measured slower here too (1.77 vs 1.57 ms at 32 q heads)
        case 8: NVX_PF(8, 8, 32, 0); break;
        default: return nvx_fail(NVX_EUNSUPPORTED, "nvx_paged_prefill: query/kv head ratio %d not in {1,2,4,8}", g);
    }
#undef NVX_PF
    return nvx_check_launch("nvx_paged_prefill");
}

}  // namespace NVX_NS
