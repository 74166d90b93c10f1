// What the two sources of nvx_softcap_attn share.
#pragma once
#include "fmt_dev.h"

namespace NVX_NS {

// position of the first key a query at `pos` sees (kept first keys aside)
__device__ __forceinline__ int first_seen(int pos, int window, int chunk) {
    if (window > 0) return pos - window + 1 > 0 ? pos - window + 1 : 0;
    return chunk > 0 ? pos - pos % chunk : 0;
}
template <typename A> __device__ __forceinline__ uint32_t cap_pack2(float lo, float hi) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef A a2 __attribute__((ext_vector_type(2)));
    const f2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, a2));
}

// The operands of nvx_softcap_attn for a ragged step without a key split (see include/nvx.h).
struct CapAttnArgs {
    const void *q, *k_cache, *v_cache;
    const int32_t* kv_indices;
    const int64_t* kv_start;
    const int32_t *kv_len, *qo_indptr;
    int n_seq, heads, kv_heads, window, chunk, keep, v_inter, gate_one, sink;
    float scale, cap, sink_score, out_mul;
    const float *r1, *r2, *slopes, *k_rn, *vcs, *sinks;
    const void* gate;
    int64_t gate_stride, out_stride;
    void* out;
};

}  // namespace NVX_NS

// 16-bit formats, heads of 128 for keys and values (with k_rn: the same rows), every operand's rows on 16-byte borders; cap_attn_mfma.hip
int nvx_softcap_attn_rows32(const NVX_NS::CapAttnArgs& args, int fmt, int64_t n_tok, hipStream_t stream);
