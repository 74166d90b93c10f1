// What the two sources of the experts' kernels share.
#pragma once
#include "fmt_dev.h"

// moe.hip: dst and src of the pairs' expert order and the experts' counts (see nvx_moe_order)
int nvx_moe_order_pairs(const int32_t* idx, int64_t n, int64_t n_exp, int64_t* dst, int32_t* src, int32_t* counts, hipStream_t stream);
// moe_gemm.hip: whether steps of many tokens go through grouped products, and the mixture as these
bool nvx_moe_grouped_fits(int fmt, int64_t n_exp, int64_t width, int64_t ff);
int nvx_moe_grouped(const void* h, int64_t h_stride, int fmt, const int32_t* idx, const float* wts, int64_t top, const void* w_gu, const void* w_d,
                    int64_t n_exp, float limit, float alpha, float shift, int weight_out, float* ws, void* out, int64_t n_tok, int64_t width, int64_t ff,
                    hipStream_t stream);
