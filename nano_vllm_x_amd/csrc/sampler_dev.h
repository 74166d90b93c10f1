// Noise and winner keys of the Gumbel-max draw, shared by the sampler (sampler.hip) and by the LM head that draws as it
// computes its logits (lmhead_sample.hip): both must give the same token for the same logits, seed and step.
#pragma once
#include "nvx_dev.h"

namespace NVX_NS {

// a * b, both halves by one instruction: a 32-bit multiply takes four times a vector instruction's time, and the generator is 20 products
__device__ __forceinline__ uint64_t mul_wide(uint32_t a, uint32_t b) {
    uint64_t d, carry;
    asm("v_mad_u64_u32 %0, %1, %2, %3, 0" : "=v"(d), "=s"(carry) : "s"(a), "v"(b));
    return d;
}

__device__ __forceinline__ uint4 philox4x32_10(uint4 ctr, uint2 key) {
    const uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = mul_wide(M0, ctr.x), p1 = mul_wide(M1, ctr.z);
        ctr = make_uint4((uint32_t)(p1 >> 32) ^ ctr.y ^ key.x, (uint32_t)p1, (uint32_t)(p0 >> 32) ^ ctr.w ^ key.y, (uint32_t)p0);
        key.x += W0; key.y += W1;
    }
    return ctr;
}

// __logf for arguments that are neither denormal, nor zero, infinite or NaN: the base-two logarithm times ln 2 in two parts, without the steps that scale
// denormals and pass infinities on (half of its instructions, and the draw is two logarithms a token)
__device__ __forceinline__ float log_of_normal(float x) {
    const float y = __builtin_amdgcn_logf(x), c = __uint_as_float(0x3f317217u), cc = __uint_as_float(0x3377d1cfu);
    return __builtin_fmaf(y, c, __builtin_fmaf(y, cc, __builtin_fmaf(y, c, -(y * c))));
}

// Gumbel noise from 23 random bits.  (r >> 9) + 0.5 is exact in fp32 (24 significant bits), so u lies
// strictly inside (0, 1); with 24 bits the top value rounds to u = 1, -log(u) = 0 and the noise becomes
// +infinity: that token would win whatever its logit.  The inner logarithm is clamped at 2^-25 as well, in
// case the fast logarithm returns 0 just below 1 (the noise is then at most 17.3).
__device__ __forceinline__ float gumbel_from_bits(uint32_t r) {
    const float u = ((float)(r >> 9) + 0.5f) * (1.0f / 8388608.0f);
    return -log_of_normal(fmaxf(-log_of_normal(u), 2.98023224e-8f));
}

// order-preserving map fp32 -> uint32 (ascending)
__device__ __forceinline__ uint32_t order_key(float x) {
    const uint32_t u = __float_as_uint(x);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// (score, token) as one 64-bit key: larger score wins, then the lower token id
__device__ __forceinline__ unsigned long long pack_winner(float v, int idx) {
    return ((unsigned long long)order_key(v) << 32) | (unsigned long long)(0xffffffffu - (uint32_t)idx);
}

}  // namespace NVX_NS
