// The layers of a Qwen3 decode step of up to eight sequences as ONE launch: from the attention of the first layer to SiluAndMul of the last.
//
// With so few rows a layer of launches is 28 to 31 us, 18 more than its weights and keys take to arrive: every launch pays its start and a trip to memory before
// its first multiplication.  Here 128 workgroups stay for the whole step; each keeps the rows of every weight that are its own and asks for them up to a
// layer ahead, so what stands between two products is only the passing on of their results.  Bound by that: 16.5 us a layer of one row, six hand-overs, 13.7 of
// them where the weights stand still.  Qwen3-0.6B, us a step, layers of launches and now: 1 sequence of 40 / 333 / 1900 tokens 787 / 867 / 915 -> 531 / 552 / 590; 2 of 300-900 887
// -> 613; 4 of 100-1024 902 -> 671; 8 of 20-40 837 -> 687, of 100-1024 954 -> 848.
//
//   * A hand-over is a word of 8 bytes, 4 of data and 4 of a tag that no earlier layer or step has used since the words were zeros: data and the news of it travel together, the reader
//     asks for the very words that it needs until all of them carry the tag.  No counter, no fence, no second trip: 1.2 us among all workgroups, 0.85 among those
//     of an XCD, with nothing else going on; a launch boundary with the first trip of its loads is 4.5.  Both sides are relaxed atomics of device scope, which
//     pass by the caches that the XCDs do not share.  A second question on its way behind the first made it slower (552 -> 622: the questions wait for each other).
//   * Words that every workgroup reads are left in four copies, and a workgroup reads one (one copy 562, two 557, four 553).  256 workgroups were no faster than
//     128 (15.7 us a layer of hand-overs and weights either way), and 128 leave room on the chip for a second launch like this one.
//   * A wave's loads, and nearly a CU's, return in order, so a question behind a stretch of weights waits for them.  The weights are asked for in pieces: two
//     loads a wave when a phase's words are there, three or four behind the words that the phase itself leaves (all of them there 569, more of them early 566).
//   * The products are those of decode_boundary.hip: eight waves share K in blocks of 64 columns and meet in LDS in the same order, so a row's result has
//     the bits that larger batches get.  The residual stays in the registers of the wave that adds to it.
//   * Attention: workgroup g has head g % 8, so that a head's projections, chunks and read-outs stay within what is one XCD here, and chunk g / 8 of the step's rows;
//     chunks are as short as 16 for all rows allow, so long rows get more of them.  The first 64 keys and values of a chunk are on their way before the queries exist.
//
// Built for these sizes in bfloat16 alone (ops.DecodeChain.fits): which rows of which weight a workgroup keeps, in LDS or in registers, is laid out for them and fills both.
//
// Every wait ends: a word that does not come within `ticks` of the wall clock makes the wave stop waiting for the rest of the launch.  Nothing that such a launch
// leaves passes for a result: its workgroup ends with NaN for every row, marks the words as no longer good (launches queued behind this one find that and end the
// same way), and raises the status word on the host, which computes the steps whose ids nobody has yet again, launch by launch (ModelRunner).
// What a wait is for is another workgroup of the same launch, so all 128 have to be on the chip at
// once; the host asks the device for twice that room (nvx_internal_decode_chain_fits) and lets no more than two go side by side, of all processes that share a network
// namespace (ops.DecodeChain, core/device_places.py); others that hold the chip longer than `ticks` are what the clock is for.
#include "nvx_dev.h"
#include "rope_dev.h"

namespace NVX_NS {

constexpr int DC_WGS = 128, DC_WAVES = 8, DC_ROWS = 8, DC_LAYERS = 32, DC_CHUNKS = 16, DC_COPIES = 4, DC_TILE = 64;
constexpr int DC_H = 1024, DC_HQ = 16, DC_HKV = 8, DC_FF = 3072, DC_QKV = (DC_HQ + 2 * DC_HKV) * 128, DC_AW = DC_HQ * 128;
static_assert(DC_CHUNKS * DC_HKV == DC_WGS && DC_HQ == 2 * DC_HKV, "a workgroup is a kv head and a chunk");
constexpr int DC_PART = 130;            // words of a chunk's result for one query head: 128 sums, the largest score, the sum of the weights

enum { DC_O, DC_N2, DC_GATE_UP, DC_DOWN, DC_N1, DC_QKV_W, DC_NQ, DC_NK, DC_K, DC_V, DC_PLACES };      // of a layer; N1 and QKV_W: the next one's
struct DcArgs {
    uint64_t layer[DC_LAYERS][DC_PLACES];
    int layers, rows;
    const uint16_t *qkv, *residual;     // of the first layer: (rows, 4096), (rows, 1024)
    uint16_t *act, *residual_out;       // of the last: (rows, 3072), (rows, 1024)
    const int64_t *positions, *kv_start, *out_slots;
    const int32_t *kv_len, *kv_indices;
    const float* cos_sin;
    int64_t max_pos, n_slots;
    unsigned long long* words;
    unsigned* epoch;                    // the first tag of the step, and whether a launch has given up (then every wait of a later one has run out as it starts)
    int* status;
    long long ticks;
    float eps, scale_log2;
};
// places of the words: two products' results with the squares of their rows, read-outs, activations (four copies each), projections, chunks
constexpr int DC_X = DC_ROWS * DC_H / 2, DC_SQ = DC_ROWS * DC_H / 8, DC_ATT = DC_ROWS * DC_AW / 2, DC_ACT = DC_ROWS * DC_FF / 2;
constexpr int DC_COPY = 2 * (DC_X + DC_SQ) + DC_ATT + DC_ACT;
constexpr int DC_QKV_AT = DC_COPIES * DC_COPY, DC_PART_AT = DC_QKV_AT + DC_ROWS * DC_QKV / 2, DC_WORDS = DC_PART_AT + DC_WGS * 2 * DC_PART;
constexpr int DC_X1 = 0, DC_SQ1 = DC_X, DC_X2 = DC_X + DC_SQ, DC_SQ2 = 2 * DC_X + DC_SQ, DC_ATT_AT = 2 * (DC_X + DC_SQ), DC_ACT_AT = DC_ATT_AT + DC_ATT;

typedef unsigned long long dc_word;
// (a base that all lanes share and 32 bits of offset: registers are what this kernel is short of)
// and global memory by name: from a table's numbers the compiler takes an address for any kind, LDS among them, and every wait for LDS waits for the load as well
template <class T>
using dc_global = __attribute__((address_space(1))) T;
template <class T>
__device__ __forceinline__ dc_global<T>* dc_at(T* base, unsigned i) { return reinterpret_cast<dc_global<T>*>(reinterpret_cast<uint64_t>(base) + (uint64_t)(i * (unsigned)sizeof(T))); }
typedef __attribute__((ext_vector_type(2))) unsigned int dc_u32x2;
template <class T>
__device__ __forceinline__ uint2 dc_get2(dc_global<T>* p) {
    const dc_u32x2 v = *reinterpret_cast<dc_global<const dc_u32x2>*>(p);
    return make_uint2(v[0], v[1]);
}
template <class V, class T>
__device__ __forceinline__ V dc_get_once(dc_global<T>* p) { return __builtin_nontemporal_load(reinterpret_cast<dc_global<const V>*>(p)); }
template <class V, class T>
__device__ __forceinline__ void dc_put(dc_global<T>* p, V v) { *reinterpret_cast<dc_global<V>*>(p) = v; }
__device__ __forceinline__ dc_word dc_load(const dc_word* words, unsigned at) { return __hip_atomic_load(dc_at(words, at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void dc_store(dc_word* words, unsigned at, unsigned tag, unsigned v) {
    __hip_atomic_store(dc_at(words, at), ((dc_word)tag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// a value that the compiler takes for a new one each time: what is computed from it is not kept in registers over the layers (a hundred addresses otherwise)
__device__ __forceinline__ unsigned dc_again(unsigned v) {
    asm volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ dc_word* dc_again(dc_word* p) {              // (the same for all lanes)
    asm volatile("" : "+s"(p));
    return p;
}

struct DcWait { long long deadline; bool dead; };
// v[i] = the data of the words base(i) + at(i) (base: of the wave, at: of the lane), of every lane of the wave that wants them, once all of them carry the tag
template <int N, class Base, class At, class Wants>
__device__ __forceinline__ void dc_poll(unsigned (&v)[N], Base base, At at, Wants wants, unsigned tag, DcWait& w) {
    for (unsigned turn = 0; !w.dead; ++turn) {
        dc_word x[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            x[i] = (dc_word)tag << 32;
            if (wants(i)) x[i] = dc_load(base(i), at(i));
        }
        bool there = true;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            v[i] = (unsigned)x[i];
            there &= (unsigned)(x[i] >> 32) == tag;
        }
        if (__all(there)) return;
        __builtin_amdgcn_s_sleep(1);
        if ((turn & 255) == 255 && wall_clock64() > w.deadline) w.dead = true;
    }
}

// This wave's part of ROWS rows of a weight, K in blocks of 64 columns, block `wave` and every eighth from there, in operand order
template <int TILES, int K>
struct DcWeight { nvx_u32x4 r[TILES][K / 256]; };
template <int I0, int I1, int TILES, int K, class Row>                   // loads I0 .. I1 - 1 of it, K / 256 a tile
__device__ __forceinline__ void dc_fetch(DcWeight<TILES, K>& w, const uint16_t* base, Row row, int wave, int lane) {
    unsigned at[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) at[t] = dc_again((unsigned)(row(t, lane & 15) * K + (lane >> 4) * 16));
#pragma unroll
    for (int i = I0; i < I1; ++i) {
        const int t = i / (K / 256), s = i % (K / 256);
        w.r[t][s] = dc_get_once<nvx_u32x4>(dc_at(base + wave * 64 + (s >> 1) * 512 + (s & 1) * 8, at[t]));
    }
}

// The same of eight rows, in LDS, 1 KB a block: half a tile of the matrix instruction, in registers it would be loaded and kept twice.  The wave that asked reads it,
// behind a wait for all of its loads.  Row r has its piece of eight columns c at place c ^ r.
constexpr int DC_LDS_BLOCKS = (DC_AW + DC_FF) / 64 / DC_WAVES, DC_WD_AT = DC_AW / 64 / DC_WAVES;
template <int B0, int B1, int K>
__device__ __forceinline__ void dc_fetch_lds(unsigned lds, const uint16_t* base, int wave, int lane) {
    const unsigned at = dc_again((unsigned)((lane >> 3) * K + ((lane & 7) ^ (lane >> 3)) * 8));
#pragma unroll
    for (int b = B0; b < B1; ++b) {
        const dc_global<const uint16_t>* g = dc_at(base + wave * 64 + b * 512, at);
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" : : "v"(g), "s"(lds + b * 1024) : "memory");
    }
}

// A wave's columns of the rows of x in LDS, 64 of a block side by side; 4 words apart from a multiple of 32, so that the rows of an operand lie in different banks
constexpr int DC_XS = DC_FF / 16 + 4;
// words of x (rows, K / 2) to LDS, and with SQUARES, in the same wait, the squares of row `wave`, added up as decode_boundary.hip adds them, to `squares_of`
template <int MR, int K, bool SQUARES>
__device__ __forceinline__ void dc_take(unsigned (*xs)[DC_XS], dc_word* words, int in, float* squares_of, int squares, int rows, unsigned tag, DcWait& w, int wave, int lane) {
    words = dc_again(words);
    constexpr int W = K / 1024, AT_ONCE = MR < 12 / W ? MR : (W == 1 ? 8 : 4), N = AT_ONCE * W;
    static_assert(!SQUARES || AT_ONCE == MR, "one wait for both");
#pragma unroll
    for (int r0 = 0; r0 < MR; r0 += AT_ONCE) {
        unsigned v[N + (SQUARES ? 2 : 0)];
        // (word q = 64 (i % W) + lane of the wave's: block wave + 8 (q / 32))
        const unsigned at = dc_again((wave + 8 * (lane >> 5)) * 32 + (lane & 31)), at_sq = dc_again(2 * lane);
        dc_poll(v, [&](int i) { return i < N ? words + in + (r0 + i / W) * (K / 2) + i % W * 512 : words + squares + wave * (DC_H / 8) + i - N; },
                [&](int i) { return i < N ? at : at_sq; }, [&](int i) { return i < N ? MR == 1 || r0 + i / W < rows : wave < rows; }, tag, w);
#pragma unroll
        for (int i = 0; i < N; ++i) xs[r0 + i / W][i % W * 64 + lane] = v[i];
        if constexpr (SQUARES) {
            float ss = quarter_sum(__uint_as_float(v[N]) + __uint_as_float(v[N + 1]));
            ss += xor16(ss);
            ss += xor32(ss);
            if (wave < rows && lane == 0) squares_of[wave] = ss;
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");                  // this wave's rows of the weights are there as well, in LDS behind the compiler's back
}
// a tile's sums of a wave, of MR rows of x: lane (quad, row)
template <int MR>
struct DcPart { nvx_f32x4 w[DC_WAVES][4 * MR]; };
template <int MR>
__device__ __forceinline__ void dc_leave(DcPart<MR>& p, nvx_f32x4 acc, int wave, int lane) {
    if ((lane & 15) < MR) p.w[wave][(lane >> 4) * MR + (lane & 15)] = acc;
}
template <int MR>
__device__ __forceinline__ nvx_f32x4 dc_sum(const DcPart<MR>& p, int lane) {      // (in order, as decode_boundary.hip; lanes of rows past MR repeat others)
    const int at = (lane >> 4) * MR + (lane & (MR - 1));
    nvx_f32x4 v[DC_WAVES];
#pragma unroll
    for (int i = 0; i < DC_WAVES; ++i) v[i] = p.w[i][at];
    nvx_f32x4 s = v[0];
#pragma unroll
    for (int i = 1; i < DC_WAVES; ++i) s += v[i];
    return s;
}
template <int MR, int TILES, int K>
__device__ __forceinline__ void dc_multiply(const DcWeight<TILES, K>& w, const unsigned (*xs)[DC_XS], DcPart<MR>* part, int wave, int lane) {
    const unsigned* x = xs[lane & (MR - 1)] + (lane >> 4) * 8;          // (rows of x past MR repeat the first ones: their results are not used)
    nvx_f32x4 acc[TILES];
    nvx_u32x4 b[K / 256];
#pragma unroll
    for (int s = 0; s < K / 256; ++s) b[s] = *reinterpret_cast<const nvx_u32x4*>(x + (s >> 1) * 32 + (s & 1) * 4);
#pragma unroll
    for (int t = 0; t < TILES; ++t) acc[t] = nvx_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < K / 256; ++s)
#pragma unroll
        for (int t = 0; t < TILES; ++t) acc[t] = mfma_16x16x32_h16(w.r[t][s], b[s], acc[t]);
#pragma unroll
    for (int t = 0; t < TILES; ++t) dc_leave<MR>(part[t], acc[t], wave, lane);
}
template <int MR, int K>
__device__ __forceinline__ void dc_multiply_lds(unsigned lds, const unsigned (*xs)[DC_XS], DcPart<MR>& part, int wave, int lane) {
    typedef __attribute__((address_space(3))) const nvx_u32x4 lds_u4;
    const unsigned* x = xs[lane & (MR - 1)] + (lane >> 4) * 8;
    const unsigned r = lane & 7, q2 = (lane >> 4) * 2;
    constexpr int N = K / 256;
    nvx_u32x4 a[N], b[N];
#pragma unroll
    for (int s = 0; s < N; ++s) {
        a[s] = *reinterpret_cast<lds_u4*>((uintptr_t)(lds + (s >> 1) * 1024 + r * 128 + ((q2 + (s & 1)) ^ r) * 16));
        b[s] = *reinterpret_cast<const nvx_u32x4*>(x + (s >> 1) * 32 + (s & 1) * 4);
    }
    nvx_f32x4 acc = nvx_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < N; ++s) acc = mfma_16x16x32_h16(a[s], b[s], acc);
    dc_leave<MR>(part, acc, wave, lane);
}

// A wave's eight tokens of a tile: of the keys eight lanes a token, lane l of them the dimensions 8 l .. 8 l + 7 and 64 from there; of the values every
// lane two dimensions of each token, so that their sums never leave the lane
struct DcTile { nvx_u32x4 k[2]; unsigned v[8]; unsigned long long ok; };      // ok: of the lanes, whether their token is there
__device__ __forceinline__ void dc_tile(DcTile& t, int slot, const uint16_t* k, const uint16_t* v, int64_t n_slots, int head, int lane) {
    const bool ok = slot >= 0 && (int64_t)slot < n_slots;
    t.ok = __ballot(ok);
    slot = ok ? slot : 0;
    const uint16_t* kr = k + head * 128 + ((int64_t)slot << 10) + (lane & 7) * 8;
    static_assert(DC_HKV * 128 == 1 << 10, "a row");
#pragma unroll
    for (int h = 0; h < 2; ++h) t.k[h] = dc_get_once<nvx_u32x4>(dc_at(kr, 64 * h));
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint16_t* vr = v + head * 128 + ((int64_t)__builtin_amdgcn_readlane(slot, 8 * j) << 10);
        t.v[j] = dc_get_once<unsigned>(dc_at(vr, (unsigned)(2 * lane)));
    }
}
__device__ __forceinline__ float dc_xor8(float v) { return dpp_move<0x128>(v); }      // row_ror:8
struct DcSoftmax { float m[2], l[2], acc[2][2]; };                      // m: the wave's, l: of the lane's tokens, acc: of the lane's dimensions
__device__ __forceinline__ float dc_dot(const nvx_u32x4 (&q)[2], const nvx_u32x4 (&k)[2]) {      // in all of a token's eight lanes
    float d = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const unsigned qw = q[h][w], kw = k[h][w];
            d = dot2_h16(qw, kw, d);
        }
    d += dpp_move<0xB1>(d);
    d += dpp_move<0x4E>(d);
    return d + dpp_move<0x141>(d);
}
__device__ __forceinline__ float dc_lane(float v, int lane) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane)); }
__device__ __forceinline__ void dc_fold(DcSoftmax& a, const DcTile& t, const nvx_u32x4 (&q)[2][2], float scale_log2, int lane) {
    float p[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        const float d = dc_dot(q[g], t.k), s = t.ok >> lane & 1 ? d * scale_log2 : -INFINITY;
        float m = fmaxf(s, dc_xor8(s));
        m = fmaxf(m, xor16(m));
        m = fmaxf(a.m[g], fmaxf(m, xor32(m)));
        const float ref = m == -INFINITY ? 0.f : m, alpha = __builtin_amdgcn_exp2f(a.m[g] - ref);
        p[g] = __builtin_amdgcn_exp2f(s - ref);
        a.m[g] = m;
        a.l[g] = a.l[g] * alpha + p[g];
        a.acc[g][0] *= alpha;
        a.acc[g][1] *= alpha;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const unsigned v = t.ok >> 8 * j & 1 ? t.v[j] : 0u;      // (a weight of zero times a stale NaN would be NaN)
        const float lo = h16lo_to_f32(v), hi = h16hi_to_f32(v);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const float w = dc_lane(p[g], 8 * j);
            a.acc[g][0] += w * lo;
            a.acc[g][1] += w * hi;
        }
    }
}

template <int MR>
__global__ __launch_bounds__(DC_WAVES * 64, 1) void decode_chain_kernel(const DcArgs a) {
    __shared__ uint64_t layer[DC_LAYERS][DC_PLACES];
    __shared__ __align__(16) unsigned xs_all[DC_WAVES][MR][DC_XS];
    __shared__ DcPart<MR> part[4];                                      // of the products with eight rows a workgroup, of the others
    __shared__ __align__(16) unsigned char weights[DC_WAVES][DC_LDS_BLOCKS * 1024];
    __shared__ __align__(16) unsigned heads[4][64];                     // two query heads, the new key, the new value
    __shared__ __align__(16) float meet[2][DC_WAVES][128], meet_m[2][DC_WAVES], meet_l[2][DC_WAVES];
    __shared__ float squares_of[MR];
    __shared__ __align__(16) float angles[128];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4, g = blockIdx.x;
    const int head = g & (DC_HKV - 1), item = g >> 3, rows = a.rows, layers = a.layers;
    // (the arguments lie far away: one trip for all of them instead of one a layer)
    for (int i = threadIdx.x; i < layers * DC_PLACES; i += DC_WAVES * 64) (&layer[0][0])[i] = (&a.layer[0][0])[i];
    const auto place = [&](int l, int which) {
        const uint64_t p = layer[l][which];
        return reinterpret_cast<uint16_t*>((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(p >> 32)) << 32 | (unsigned)__builtin_amdgcn_readfirstlane((int)p));
    };
    const dc_word state = __hip_atomic_load(reinterpret_cast<dc_word*>(a.epoch), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned epoch = (unsigned)state;
    DcWait wait = {wall_clock64() + a.ticks, (state >> 32) != 0};
    // ---- the chunks: the shortest length, a multiple of 64, that leaves at most 16 of them ----------------------------------------------------------
    int chunk;
    {
        long long total = 0;
        for (int r = 0; r < rows; ++r) total += max(a.kv_len[r], 0);
        const int least = max(1, (int)((total + DC_CHUNKS * DC_TILE - 1) / (DC_CHUNKS * DC_TILE)));
        const int most = max(1, (int)((total + (DC_CHUNKS - DC_ROWS) * DC_TILE - 1) / ((DC_CHUNKS - DC_ROWS) * DC_TILE))), step = (most - least + 62) / 63;
        const int c = (least + lane * step) * DC_TILE;                  // (lane 63: at least `most`, which always does)
        int n = 0;
        for (int r = 0; r < rows; ++r) n += max(1, (int)(((long long)max(a.kv_len[r], 0) + c - 1) / c));
        chunk = __builtin_amdgcn_readlane(c, __ffsll((long long)__ballot(n <= DC_CHUNKS)) - 1);
    }
    int row = -1, from = 0, count = 0;                                  // of this workgroup's chunk; `row` -1: there is none
    bool last = false;
    int merge_first = 0, merge_chunks = 0;                              // of the row whose chunks this wave joins
    {
        int first = 0;
        for (int r = 0; r < rows; ++r) {
            const int len = max(a.kv_len[r], 0), n = max(1, (int)(((long long)len + chunk - 1) / chunk));
            if (item >= first && item < first + n) {
                row = r;
                from = (item - first) * chunk;
                count = min(chunk, len - from);
                last = item == first + n - 1;
            }
            if (r == wave) { merge_first = first; merge_chunks = n; }
            first += n;
        }
    }
    const int64_t new_slot = row >= 0 && last && count > 0 ? a.out_slots[row] : -1;
    const bool own_new = new_slot >= 0 && new_slot < a.n_slots;
    const int pool = own_new ? count - 1 : count;                       // the new token's row is made here
    const int32_t* slots = a.kv_indices + (row >= 0 ? a.kv_start[row] + from : 0);
    const int token = wave * 8 + (lane >> 3);
    const int slot0 = token < pool ? slots[token] : -1;                                      // (every layer starts with it)
    if (row >= 0 && wave == 0) {
        const float* cs = a.cos_sin + clamp_pos(a.positions[row], a.max_pos) * 128;
        *reinterpret_cast<float2*>(angles + 2 * lane) = *reinterpret_cast<const float2*>(cs + 2 * lane);
    }
    // ---- this workgroup's rows of the weights, and the residual of its columns (wave 0; the upper half of the lanes for copies 2 and 3) ---------------
    const unsigned lds = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)weights[wave];
    // rows of qkv that make this head's queries, keys and values
    const int qkv_row = (item < 8 ? head * 256 : item < 12 ? (DC_HQ + head) * 128 - 256 : (DC_HQ + DC_HKV + head) * 128 - 384) + item * 32;
    const auto qkv_rows = [&](int t, int l) { return qkv_row + t * 16 + l; };
    const auto gate_rows = [&](int t, int l) { return (l & 8 ? DC_FF : 0) + g * 24 + t * 8 + (l & 7); };      // eight gate rows, the up rows beside them
    const int col = g * 8 + (quad & 1) * 4, er = l16 < MR ? min(l16, rows - 1) : 0;
    const bool live = l16 < MR && l16 < rows;
    uint2 res = *reinterpret_cast<const uint2*>(a.residual + (int64_t)er * DC_H + col);
    __syncthreads();
    DcWeight<3, DC_H> wg;
    DcWeight<2, DC_H> wq;
    DcTile tile;
    dc_tile(tile, slot0, place(0, DC_K), place(0, DC_V), a.n_slots, head, lane);
    dc_fetch_lds<0, 4, DC_AW>(lds, place(0, DC_O) + g * 8 * DC_AW, wave, lane);
    dc_fetch<0, 8>(wg, place(0, DC_GATE_UP), gate_rows, wave, lane);
    unsigned (*xs)[DC_XS] = xs_all[wave];
    dc_word* words = a.words;
    const int copy = (g >> 3) % DC_COPIES * DC_COPY;
    // a product + residual, times the next norm's weight, and the squares: wave 0
    auto leave = [&](uint2 nw, int x_at, int sq_at, unsigned tag) {
        const unsigned mine = dc_again((quad >> 1) * 2 * DC_COPY + l16 * (DC_H / 2)), mine_sq = dc_again((quad >> 1) * 2 * DC_COPY + l16 * (DC_H / 8));
        const nvx_f32x4 s = dc_sum<MR>(part[0], lane);
        const float v[4] = {round_h16(s[0]) + h16lo_to_f32(res.x), round_h16(s[1]) + h16hi_to_f32(res.x), round_h16(s[2]) + h16lo_to_f32(res.y), round_h16(s[3]) + h16hi_to_f32(res.y)};
        float sq = v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        sq += xor16(sq);
        res = make_uint2(pack_h16x2(v[0], v[1]), pack_h16x2(v[2], v[3]));
        const unsigned y0 = pack_h16x2(v[0] * h16lo_to_f32(nw.x), v[1] * h16hi_to_f32(nw.x)), y1 = pack_h16x2(v[2] * h16lo_to_f32(nw.y), v[3] * h16hi_to_f32(nw.y));
        if (live) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                dc_word* to = words + c * DC_COPY + x_at + g * 4;
                dc_store(to, mine + (quad & 1) * 2, tag, y0);
                dc_store(to + 1, mine + (quad & 1) * 2, tag, y1);
                if (!(quad & 1)) dc_store(words + c * DC_COPY + sq_at + g, mine_sq, tag, __float_as_uint(sq));
            }
        }
    };
    uint2 nw1 = {}, nw2 = {}, hw[2] = {};                               // wave 0: the norms' weights of a layer, asked for in the layer before
    const auto norms = [&](int l) {
        nw2 = dc_get2(dc_at(place(l, DC_N2), col));
        if (l + 1 < layers) nw1 = dc_get2(dc_at(place(l, DC_N1), col));
        const uint16_t* w = quad < 2 ? place(l, DC_NQ) : place(l, DC_NK);
        hw[0] = dc_get2(dc_at(w, 4 * l16));
        hw[1] = dc_get2(dc_at(w, 64 + 4 * l16));
    };
    if (wave == 0) norms(0);
    for (int l = 0; l < layers; ++l) {
        const unsigned tag = epoch + l;
        const bool more = l + 1 < layers;
        words = dc_again(words);
        // ---- queries, the new key and value ---------------------------------------------------------------------------------------------------------
        if (row >= 0 && wave == 0) {                                    // quarter-waves: two query heads, key, value
            const int at = (quad < 2 ? head * 2 + quad : quad == 2 ? DC_HQ + head : DC_HQ + DC_HKV + head) * 128;
            unsigned x[4];
            if (l == 0) {
                const uint16_t* p = a.qkv + (int64_t)row * DC_QKV + at + 4 * l16;
                const uint2 lo = *reinterpret_cast<const uint2*>(p), hi = *reinterpret_cast<const uint2*>(p + 64);
                x[0] = lo.x; x[1] = lo.y; x[2] = hi.x; x[3] = hi.y;
            } else {
                const unsigned from_at = dc_again(at / 2 + 2 * l16);
                dc_poll(x, [&](int i) { return words + DC_QKV_AT + row * (DC_QKV / 2) + (i & 1) + (i >> 1) * 32; }, [&](int) { return from_at; }, [](int) { return true; },
                        tag - 1, wait);
            }
            HalfQuad h;
            h.a[0] = h16lo_to_f32(x[0]); h.a[1] = h16hi_to_f32(x[0]); h.a[2] = h16lo_to_f32(x[1]); h.a[3] = h16hi_to_f32(x[1]);
            h.b[0] = h16lo_to_f32(x[2]); h.b[1] = h16hi_to_f32(x[2]); h.b[2] = h16lo_to_f32(x[3]); h.b[3] = h16hi_to_f32(x[3]);
            const uint4 o = norm_rotate_interleave(h, half_quad_sumsq(h), hw[0], hw[1], a.eps, angles, l16);
            if (quad < 3) *reinterpret_cast<uint4*>(&heads[quad][4 * l16]) = o;
            else { heads[3][2 * l16] = x[0]; heads[3][2 * l16 + 1] = x[1]; heads[3][32 + 2 * l16] = x[2]; heads[3][33 + 2 * l16] = x[3]; }
        }
        __syncthreads();
        // ---- attention of the chunk -----------------------------------------------------------------------------------------------------------------
        if (row >= 0) {
            nvx_u32x4 q[2][2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) q[i][h] = *reinterpret_cast<const nvx_u32x4*>(&heads[i][(lane & 7) * 4 + 32 * h]);
            DcSoftmax sm = {{-INFINITY, -INFINITY}, {0.f, 0.f}, {{0.f, 0.f}, {0.f, 0.f}}};
            int slot = DC_TILE + token < pool ? slots[DC_TILE + token] : -1;
            for (int t0 = 0; t0 < pool; t0 += DC_TILE) {
                const DcTile now = tile;
                if (t0 + DC_TILE < pool) {
                    dc_tile(tile, slot, place(l, DC_K), place(l, DC_V), a.n_slots, head, lane);
                    const int t = t0 + 2 * DC_TILE + token;
                    slot = t < pool ? slots[t] : -1;
                }
                dc_fold(sm, now, q, a.scale_log2, lane);
            }
            if (own_new && wave == 0) {
                nvx_u32x4 k[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) k[h] = *reinterpret_cast<const nvx_u32x4*>(&heads[2][(lane & 7) * 4 + 32 * h]);
                const unsigned v = heads[3][lane];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const float s = dc_dot(q[i], k) * a.scale_log2, m = fmaxf(sm.m[i], s), ref = m == -INFINITY ? 0.f : m;
                    const float alpha = __builtin_amdgcn_exp2f(sm.m[i] - ref), p = __builtin_amdgcn_exp2f(s - ref);
                    sm.m[i] = m;
                    sm.l[i] = sm.l[i] * alpha + (lane < 8 ? p : 0.f);
                    sm.acc[i][0] = sm.acc[i][0] * alpha + p * h16lo_to_f32(v);
                    sm.acc[i][1] = sm.acc[i][1] * alpha + p * h16hi_to_f32(v);
                }
                if (lane < 16) {
                    const int64_t at = (new_slot * DC_HKV + head) * 128 + 8 * lane;
                    dc_put(dc_at(place(l, DC_K) + at, 0), *reinterpret_cast<const nvx_u32x4*>(&heads[2][4 * lane]));
                    dc_put(dc_at(place(l, DC_V) + at, 0), *reinterpret_cast<const nvx_u32x4*>(&heads[3][4 * lane]));
                }
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                float sum = sm.l[i];
                sum += dc_xor8(sum);
                sum += xor16(sum);
                sum += xor32(sum);
                *reinterpret_cast<float2*>(&meet[i][wave][2 * lane]) = make_float2(sm.acc[i][0], sm.acc[i][1]);
                if (lane == 0) { meet_m[i][wave] = sm.m[i]; meet_l[i][wave] = sum; }
            }
        }
        __syncthreads();
        if (row >= 0 && wave < 4) {
            const int i = wave >> 1, d = (wave & 1) * 64 + lane;
            float mw[DC_WAVES], lw[DC_WAVES], m = -INFINITY, o = 0.f, sum = 0.f;
#pragma unroll
            for (int w = 0; w < DC_WAVES; w += 4) {
                *reinterpret_cast<float4*>(mw + w) = *reinterpret_cast<const float4*>(&meet_m[i][w]);
                *reinterpret_cast<float4*>(lw + w) = *reinterpret_cast<const float4*>(&meet_l[i][w]);
            }
#pragma unroll
            for (int w = 0; w < DC_WAVES; ++w) m = fmaxf(m, mw[w]);
            const float ref = m == -INFINITY ? 0.f : m;
#pragma unroll
            for (int w = 0; w < DC_WAVES; ++w) {
                const float s = __builtin_amdgcn_exp2f(mw[w] - ref);
                o += s * meet[i][w][d];
                sum += s * lw[w];
            }
            dc_word* to = words + DC_PART_AT + (g * 2 + i) * DC_PART;
            dc_store(to, d, tag, __float_as_uint(o));
            if (d == 0) {
                dc_store(to, 128, tag, __float_as_uint(m));
                dc_store(to, 129, tag, __float_as_uint(sum));
            }
        }
        const uint16_t* const w_down = place(l, DC_DOWN) + g * 8 * DC_FF;
        __syncthreads();                                                // (behind the words that the step waits for)
        dc_fetch<8, 12>(wg, place(l, DC_GATE_UP), gate_rows, wave, lane);
        dc_fetch_lds<0, 1, DC_FF>(lds + DC_WD_AT * 1024, w_down, wave, lane);
        // ---- the chunks of a row meet: 16 dimensions of a query head a workgroup, a row a wave, four chunks side by side ---------------------------------
        if (wave < rows) {
            const int qh = 2 * head + (item >> 3), dims = (item & 7) * 16;
            const dc_word* mine = words + DC_PART_AT + ((merge_first * DC_HKV + (qh >> 1)) * 2 + (qh & 1)) * DC_PART;
            float m[4], s[4], o[4], mx = -INFINITY;
            unsigned v[12];
            const unsigned at = dc_again(quad * (DC_HKV * 2 * DC_PART));
            dc_poll(v, [&](int i) { return mine + i / 3 * (4 * DC_HKV * 2 * DC_PART) + (i % 3 == 0 ? dims : 127 + i % 3); }, [&](int i) { return i % 3 == 0 ? at + l16 : at; },
                    [&](int i) { return i / 3 * 4 + quad < merge_chunks; }, tag, wait);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool is = 4 * j + quad < merge_chunks;
                o[j] = is ? __uint_as_float(v[3 * j]) : 0.f;
                m[j] = is ? __uint_as_float(v[3 * j + 1]) : -INFINITY;
                s[j] = is ? __uint_as_float(v[3 * j + 2]) : 0.f;
                mx = fmaxf(mx, m[j]);
            }
            mx = fmaxf(mx, xor16(mx));
            mx = fmaxf(mx, xor32(mx));
            const float ref = mx == -INFINITY ? 0.f : mx;
            float out = 0.f, sum = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float e = __builtin_amdgcn_exp2f(m[j] - ref);
                out += e * o[j];
                sum += e * s[j];
            }
            out += xor16(out);
            out += xor32(out);
            sum += xor16(sum);
            sum += xor32(sum);
            const float r = sum > 0.f ? out / sum : 0.f, next = dpp_move<0xB1>(r);
            if (!(lane & 1)) dc_store(words + DC_ATT_AT + wave * (DC_AW / 2) + qh * 64 + dims / 2, dc_again(quad * DC_COPY + (l16 >> 1)), tag, pack_h16x2(r, next));
        }
        __syncthreads();                                                // (behind the words that the step waits for)
        dc_fetch_lds<1, 6, DC_FF>(lds + DC_WD_AT * 1024, w_down, wave, lane);
        // ---- output projection ----------------------------------------------------------------------------------------------------------------------
        const uint16_t* const w_qkv = place(l, DC_QKV_W);                   // (a place is two trips to LDS and back: ahead of the waits)
        dc_take<MR, DC_AW, false>(xs, words, copy + DC_ATT_AT, squares_of, 0, rows, tag, wait, wave, lane);
        if (more) dc_fetch<0, 2>(wq, w_qkv, qkv_rows, wave, lane);
        dc_multiply_lds<MR, DC_AW>(lds, xs, part[0], wave, lane);
        __syncthreads();
        if (wave == 0) leave(nw2, DC_X1, DC_SQ1, tag);
        __syncthreads();                                                // (behind the words that the step waits for)
        if (more) dc_fetch<2, 5>(wq, w_qkv, qkv_rows, wave, lane);
        // ---- gate | up with SiluAndMul ----------------------------------------------------------------------------------------------------------------
        dc_take<MR, DC_H, true>(xs, words, copy + DC_X1, squares_of, copy + DC_SQ1, rows, tag, wait, wave, lane);
        if (more) dc_fetch<5, 7>(wq, w_qkv, qkv_rows, wave, lane);
        else wq = {};                                                   // (or the registers of the last ones would be kept for this case through the layer)
        dc_multiply<MR>(wg, xs, part + 1, wave, lane);
        __syncthreads();
        if (wave < 3) {
            const float inv = 1.0f / sqrtf(squares_of[er] / (float)DC_H + a.eps);
            const nvx_f32x4 s = dc_sum<MR>(part[1 + wave], lane);
            float o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float x = round_h16(s[i] * inv), other = xor32(x), gate = lane < 32 ? x : other, up = lane < 32 ? other : x;
                o[i] = silu_h16(gate) * up;
            }
            const unsigned y0 = pack_h16x2(o[0], o[1]), y1 = pack_h16x2(o[2], o[3]);
            const int at = g * 24 + wave * 8 + (quad & 1) * 4;
            if (more) {
                const unsigned mine = dc_again((quad >> 1) * 2 * DC_COPY + l16 * (DC_FF / 2) + (quad & 1) * 2);
                if (live) {
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        dc_word* to = words + c * DC_COPY + DC_ACT_AT + g * 12 + wave * 4;
                        dc_store(to, mine, tag, y0);
                        dc_store(to + 1, mine, tag, y1);
                    }
                }
            } else if (live && lane < 32) dc_put(dc_at(a.act, dc_again(l16 * DC_FF + at)), dc_u32x2{y0, y1});
        }
        if (!more) break;
        const uint16_t *const w_o = place(l + 1, DC_O) + g * 8 * DC_AW, *const w_gate_up = place(l + 1, DC_GATE_UP);
        __syncthreads();                                                // (behind the words that the step waits for)
        dc_fetch<7, 8>(wq, w_qkv, qkv_rows, wave, lane);
        dc_fetch_lds<0, 2, DC_AW>(lds, w_o, wave, lane);
        if (pool > 0) dc_tile(tile, slot0, place(l + 1, DC_K), place(l + 1, DC_V), a.n_slots, head, lane);
        else tile = {};
        // ---- down projection --------------------------------------------------------------------------------------------------------------------------
        dc_take<MR, DC_FF, false>(xs, words, copy + DC_ACT_AT, squares_of, 0, rows, tag, wait, wave, lane);
        dc_fetch_lds<2, 4, DC_AW>(lds, w_o, wave, lane);
        dc_multiply_lds<MR, DC_FF>(lds + DC_WD_AT * 1024, xs, part[0], wave, lane);
        __syncthreads();
        if (wave == 0) leave(nw1, DC_X2, DC_SQ2, tag);
        __syncthreads();                                                // (behind the words that the step waits for)
        if (wave == 0) norms(l + 1);
        dc_fetch<0, 3>(wg, w_gate_up, gate_rows, wave, lane);
        // ---- the next layer's queries, keys and values ----------------------------------------------------------------------------------------------------
        dc_take<MR, DC_H, true>(xs, words, copy + DC_X2, squares_of, copy + DC_SQ2, rows, tag, wait, wave, lane);
        dc_fetch<3, 5>(wg, w_gate_up, gate_rows, wave, lane);
        dc_multiply<MR>(wq, xs, part + 1, wave, lane);
        __syncthreads();
        if (wave < 2) {
            const float inv = 1.0f / sqrtf(squares_of[er] / (float)DC_H + a.eps);
            const nvx_f32x4 s = dc_sum<MR>(part[1 + wave], lane);
            if (live) {
                dc_word* to = words + DC_QKV_AT + qkv_row / 2 + wave * 8;
                const unsigned mine = dc_again(l16 * (DC_QKV / 2) + quad * 2);
                dc_store(to, mine, tag, pack_h16x2(s[0] * inv, s[1] * inv));
                dc_store(to + 1, mine, tag, pack_h16x2(s[2] * inv, s[3] * inv));
            }
        }
        __syncthreads();                                                // (behind the words that the step waits for)
        dc_fetch<5, 8>(wg, w_gate_up, gate_rows, wave, lane);
    }
    if (wave == 0 && live && lane < 32) dc_put(dc_at(a.residual_out, dc_again(l16 * DC_H + col)), dc_u32x2{res.x, res.y});
    if (lane == 0) meet_l[0][wave] = wait.dead ? 1.f : 0.f;
    __syncthreads();
    float gave_up = 0.f;
#pragma unroll
    for (int w = 0; w < DC_WAVES; ++w) gave_up += meet_l[0][w];
    if (gave_up != 0.f) {                                               // (24 columns of the last product's rows that are no numbers make none of every number behind it)
        for (int i = threadIdx.x; i < rows * 24; i += DC_WAVES * 64) a.act[i / 24 * DC_FF + g * 24 + i % 24] = 0x7fc0;
        if (threadIdx.x == 0) {
            __hip_atomic_store(a.epoch + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    // every workgroup has left words that this one has read since, so every one has read the epoch (or this one has given up, and no later launch goes by it)
    if (g == 0 && threadIdx.x == 0) __hip_atomic_store(a.epoch, epoch + layers, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace NVX_NS

using namespace NVX_NS;

extern "C" int64_t nvx_internal_decode_chain_words(void) { return DC_WORDS; }

// whether the current device has room for two launches at once
extern "C" int nvx_internal_decode_chain_fits(void) {
    int dev = -1, cus = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, decode_chain_kernel<DC_ROWS>, DC_WAVES * 64, 0) != hipSuccess) return 0;
    return (int64_t)cus * per >= 2 * DC_WGS;
}

// layers: per layer o, post-attention norm, gate | up, down, the next layer's input norm and qkv (the last: none), q norm, k norm, k rows, v rows.  ws: `words`
// of zeros, epoch: two ints, 1 or more and 0; both are the next call's as this one leaves them, for fewer than 2^32 / n_layers calls.  status: pinned host memory.  workgroups: 128; with fewer the waits
// for what the others would leave run out, `seconds` into the launch.
extern "C" int nvx_internal_decode_chain(const int64_t* layers, int64_t n_layers, int64_t rows, const void* qkv, const void* residual, void* act, void* residual_out,
                                         const int64_t* positions, const int64_t* kv_start, const int32_t* kv_len, const int64_t* out_slots, const int32_t* kv_indices,
                                         const float* cos_sin, int64_t max_pos, int64_t n_slots, void* ws, void* epoch, void* status, double seconds, int64_t workgroups,
                                         float eps, float sm_scale, nvx_stream_t stream) {
    NVX_REQUIRE(layers && qkv && residual && act && residual_out && positions && kv_start && kv_len && out_slots && kv_indices && cos_sin && ws && epoch && status, NVX_EINVAL,
                "nvx_internal_decode_chain: null pointer");
    NVX_REQUIRE(n_layers > 0 && n_layers <= DC_LAYERS && rows > 0 && rows <= DC_ROWS && max_pos > 0 && n_slots > 0 && seconds > 0 && seconds <= 60 && workgroups > 0 &&
                    workgroups <= DC_WGS, NVX_EUNSUPPORTED,
                "nvx_internal_decode_chain: sizes");
    DcArgs a = {};
    for (int64_t i = 0; i < n_layers; ++i) {
        const int64_t* p = layers + DC_PLACES * i;
        for (int j = 0; j < DC_PLACES; ++j) {
            NVX_REQUIRE((p[j] && p[j] % 16 == 0) || (i + 1 == n_layers && (j == DC_N1 || j == DC_QKV_W)), NVX_EINVAL, "nvx_internal_decode_chain: weights and caches must be 16-byte aligned");
            a.layer[i][j] = (uint64_t)p[j];
        }
    }
    NVX_REQUIRE(nvx_aligned16(qkv) && nvx_aligned16(residual) && nvx_aligned16(act) && nvx_aligned16(residual_out) && nvx_aligned16(cos_sin) && nvx_aligned16(ws) &&
                    (reinterpret_cast<uintptr_t>(epoch) & 7) == 0, NVX_EINVAL, "nvx_internal_decode_chain: pointers must be 16-byte aligned");
    a.layers = (int)n_layers; a.rows = (int)rows;
    a.qkv = (const uint16_t*)qkv; a.residual = (const uint16_t*)residual; a.act = (uint16_t*)act; a.residual_out = (uint16_t*)residual_out;
    a.positions = positions; a.kv_start = kv_start; a.out_slots = out_slots; a.kv_len = kv_len; a.kv_indices = kv_indices;
    a.cos_sin = cos_sin; a.max_pos = max_pos; a.n_slots = n_slots;
    a.words = (unsigned long long*)ws; a.epoch = (unsigned*)epoch; a.status = (int*)status;
    a.ticks = (long long)(seconds * 1e8);                               // the wall clock counts at 100 MHz
    a.eps = eps; a.scale_log2 = sm_scale * 1.4426950408889634f;
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((unsigned)workgroups);
    if (rows == 1) hipLaunchKernelGGL(decode_chain_kernel<1>, grid, dim3(DC_WAVES * 64), 0, st, a);
    else if (rows == 2) hipLaunchKernelGGL(decode_chain_kernel<2>, grid, dim3(DC_WAVES * 64), 0, st, a);
    else if (rows <= 4) hipLaunchKernelGGL(decode_chain_kernel<4>, grid, dim3(DC_WAVES * 64), 0, st, a);
    else hipLaunchKernelGGL(decode_chain_kernel<8>, grid, dim3(DC_WAVES * 64), 0, st, a);
    return nvx_check_launch("nvx_internal_decode_chain");
}
