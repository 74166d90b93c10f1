// The layers of a Qwen3 prefill step, queued by one call.  Host code: it launches the kernels that the module graph launches, in the
// same order, and is not part of the C ABI.
//
// Up to some thousand tokens the device needs less than 150 us for a layer and the host, through Python, 160 to queue it (220 where it calls
// modules): four library products at 19 us each, shape look-up included, and six kernels at 10.  From here a kernel is 2-4 us, and the products are
// those of prefill_gemm.hip.  Qwen3-0.6B, us a step through Python and from here: 20 tokens 4540 and 1270, 459 tokens 4560 and 1850 (6200
// through the modules); 2160 tokens behind cached ones, float16, 6270 and 4980.
#include "prefill_gemm.h"

// layers: ten addresses a layer: input norm, qkv, q norm, k norm, o, post-attention norm, gate | up, down (weights), k rows, v rows (caches).
// x (T, hidden): the embedding rows.  Workspace: h (normed rows), sum (a projection's result), res0 and res1 (residuals), (T, hidden) each; qkv
// rows; q and attn (T, hq * 128 each); act (T, inter); all in the 16-bit format.  out: the final-normed rows.
struct NvxPrefillStep {
    const int64_t* layers;
    int64_t n_layers, n_tok, batch, hidden, hq, hkv, inter, rope_rows, n_slots;
    const void *x, *final_norm;
    const int64_t *positions, *slots;
    const float* rope;
    const int32_t *qo_indptr, *kv_indptr, *kv_indices, *plan;
    void *h, *sum, *res0, *res1, *qkv, *q, *attn, *act, *out;
    double eps, scale;
};

extern "C" int NVX_ENTRY(nvx_internal_prefill_step)(const NvxPrefillStep* s, nvx_stream_t stream) {
    const int64_t t = s->n_tok, hid = s->hidden, qw = (s->hq + 2 * s->hkv) * 128, aw = s->hq * 128;
    const float eps = (float)s->eps;
    const hipStream_t st = (hipStream_t)stream;
    void* res[2] = {s->res0, s->res1};
#define NVX_STEP(call) do { if (const int rc = (call)) return rc; } while (0)
    NVX_STEP(NVX_ENTRY(nvx_rmsnorm)(s->x, hid, nullptr, (const void*)s->layers[0], 0, s->h, nullptr, t, hid, eps, stream));
    const void* residual = s->x;
    int turn = 0;
    for (int64_t l = 0; l < s->n_layers; ++l) {
        const int64_t* w = s->layers + 10 * l;
        if (NVX_ENTRY(nvx_prefill_heads_ride)(t, qw, hid)) {      // a head's norm and rotation at the end of the product (sizes and figures there)
            const NvxQkvOut out = {s->positions, s->slots, s->rope, s->rope_rows, s->n_slots, (const uint16_t*)w[2], (const uint16_t*)w[3], (uint16_t*)s->q,
                                   (uint16_t*)w[8], (uint16_t*)w[9], (int)s->hq, (int)s->hkv, eps};
            NVX_STEP(NVX_ENTRY(nvx_prefill_gemm)(s->h, hid, (const void*)w[1], nullptr, t, qw, hid, NVX_PG_QKV, &out, st));
        } else {
            NVX_STEP(NVX_ENTRY(nvx_prefill_gemm)(s->h, hid, (const void*)w[1], s->qkv, t, qw, hid, NVX_PG_PLAIN, nullptr, st));
            NVX_STEP(NVX_ENTRY(nvx_qknorm_rope_store)(s->qkv, qw, s->positions, s->rope, s->rope_rows, (const void*)w[2], (const void*)w[3], eps, s->slots, s->q,
                                                     (void*)w[8], (void*)w[9], s->n_slots, t, (int)s->hq, (int)s->hkv, stream));
        }
        NVX_STEP(NVX_ENTRY(nvx_paged_prefill)(s->q, aw, (const void*)w[8], (const void*)w[9], s->n_slots, s->qo_indptr, s->kv_indptr, s->kv_indices, s->plan,
                                             s->attn, t, s->batch, (int)s->hq, (int)s->hkv, (float)s->scale, stream));
        NVX_STEP(NVX_ENTRY(nvx_prefill_gemm)(s->attn, aw, (const void*)w[4], s->sum, t, hid, aw, NVX_PG_PLAIN, nullptr, st));
        NVX_STEP(NVX_ENTRY(nvx_rmsnorm)(s->sum, hid, residual, (const void*)w[5], 0, s->h, res[turn], t, hid, eps, stream));
        residual = res[turn];
        turn ^= 1;
        NVX_STEP(NVX_ENTRY(nvx_prefill_gemm)(s->h, hid, (const void*)w[6], s->act, t, 2 * s->inter, hid, NVX_PG_SILU, nullptr, st));
        NVX_STEP(NVX_ENTRY(nvx_prefill_gemm)(s->act, s->inter, (const void*)w[7], s->sum, t, hid, s->inter, NVX_PG_PLAIN, nullptr, st));
        const bool last = l + 1 == s->n_layers;
        NVX_STEP(NVX_ENTRY(nvx_rmsnorm)(s->sum, hid, residual, last ? s->final_norm : (const void*)w[10], 0, last ? s->out : s->h, res[turn], t, hid, eps, stream));
        residual = res[turn];
        turn ^= 1;
    }
#undef NVX_STEP
    return NVX_OK;
}
