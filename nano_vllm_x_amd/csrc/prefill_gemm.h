// The products of prefill steps (prefill_gemm.hip), for the host code that queues them.
#pragma once
#include "nvx_dev.h"

// y (m, n) = x (m, k) w (n, k)^T, or with `silu` (m, n / 2) = SiluAndMul of it, in the 16-bit format; rows of x `x_stride` elements apart
int NVX_ENTRY(nvx_prefill_gemm)(const void* x, int64_t x_stride, const void* w, void* y, int64_t m, int64_t n, int64_t k, bool silu, hipStream_t st);
