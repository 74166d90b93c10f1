// What the sources of the experts' kernels share.
#pragma once
#include "fmt_dev.h"

// What stands behind a mixture where its sums go straight on: x += r / rms(r) * w_post, h_out = x / rms(x) * w_next (nvx_postnorm_residual without a
// second result)
struct NvxMoeEnd {
    float* x;
    const float* w_post;
    int64_t w_post_n;
    const float* w_next;
    int64_t w_next_n;
    float eps;
    void* h_out;
};
// gate_norm.hip: whether a launch can take the sums with that end, and the launch
bool nvx_pairs_postnorm_fits(int fmt, const NvxMoeEnd& e, int64_t width);
int nvx_pairs_postnorm(int fmt, const float* o, const int64_t* dst, const float* wts, int64_t top, const NvxMoeEnd& e, int64_t n_tok, int64_t width,
                       hipStream_t stream);
// moe.hip: dst and src of the pairs' expert order and the experts' counts (see nvx_moe_order)
int nvx_moe_order_pairs(const int32_t* idx, int64_t n, int64_t n_exp, int64_t* dst, int32_t* src, int32_t* counts, hipStream_t stream);
// moe_gemm.hip: whether steps of many tokens go through grouped products, and the mixture as these (`end`, where given, instead of `out`)
bool nvx_moe_grouped_fits(int fmt, int64_t n_exp, int64_t width, int64_t ff);
int nvx_moe_grouped(const void* h, int64_t h_stride, int fmt, const int32_t* idx, const float* wts, int64_t top, const void* w_gu, const void* w_d,
                    int64_t n_exp, float limit, float alpha, float shift, int weight_out, float* ws, void* out, int64_t n_tok, int64_t width, int64_t ff,
                    const NvxMoeEnd* end, hipStream_t stream);
