// silu_near.h -- bf16 results of the exact SiLU and sigmoid (uzu_math.h: the exponential in 64 bits) from quick f32 quotients.
//
// What an element of a gate or a convolution costs is its exact exponential: fifteen instructions in 64 bits and a division, 200 cycles a wave.  The result is rounded to bf16,
// so a quotient that is known to a few f32 ulps decides it, unless it lies next to a tie: then, for one element in a thousand, the exact one is worked out after all.  The
// results are the same bits: silu_bf16 was compared for all 2^32 arguments (silu_conv_check.cpp of the host tests, which looks at the range where the quotient decides every time), the
// scaled forms for all bf16 gates of a norm-gate; otherwise they rest on the bound: three roundings and the exponential's 4 ulps, the reciprocal's 1 and the scale's, within 24.
#pragma once
#include "device_utils.h"
#include "uzu_math.h"

namespace uzu {
namespace k {

// e^-x within 4 f32 ulps for |x| < 80: the product with log2 e in two floats, the smaller one as a factor (its square, dropped, is below 2^-40)
__device__ __forceinline__ float exp_neg_near(float x) {
    const float a = x * -0x1.715476p+0f, rest = fmaf(x, -0x1.4ae0cp-26f, fmaf(x, -0x1.715476p+0f, -a)), e = __builtin_amdgcn_exp2f(a);
    return fmaf(e, rest * 0x1.62e43p-1f, e);
}
// bf16(y) needs the exact y: `near` (within 24 f32 ulps of it) is within 32 ulps of a tie, or the quick forms don't reach that far
__device__ __forceinline__ bool near_undecided(float x, float near) { return !(x > -80.0f && x < 80.0f) || ((f32_to_bits(near) + 0x8020u) & 0xFFFFu) <= 0x40u; }

// f32_to_bf16(silu_f32_tab(x))
__device__ __forceinline__ uint16_t silu_bf16(float x, const uint64_t* tab) {
    const float near = x * __builtin_amdgcn_rcpf(1.0f + exp_neg_near(x));
    if (__builtin_expect(near_undecided(x, near), 0)) return f32_to_bf16(silu_f32_tab(x, tab));
    return f32_to_bf16(near);
}
// f32_to_bf16(scale * silu_f32_tab(x))
__device__ __forceinline__ uint16_t scaled_silu_bf16(float scale, float x, const uint64_t* tab) {
    const float near = scale * (x * __builtin_amdgcn_rcpf(1.0f + exp_neg_near(x)));
    if (__builtin_expect(near_undecided(x, near), 0)) return f32_to_bf16(scale * silu_f32_tab(x, tab));
    return f32_to_bf16(near);
}
// f32_to_bf16(scale * (1 / (1 + e^-x)))
__device__ __forceinline__ uint16_t scaled_sigmoid_bf16(float scale, float x, const uint64_t* tab) {
    const float near = scale * __builtin_amdgcn_rcpf(1.0f + exp_neg_near(x));
    if (__builtin_expect(near_undecided(x, near), 0)) return f32_to_bf16(scale * (1.0f / (1.0f + expf_glibc_tab(-x, tab))));
    return f32_to_bf16(near);
}

} // namespace k
} // namespace uzu
