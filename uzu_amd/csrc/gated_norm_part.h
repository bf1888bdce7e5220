// gated_norm_part.h -- a part of a row through GatedNormParams' norm: the body of gated_norm_rows (k_causal_conv.hip), and of the workgroups that stand beside the merge of a
// decode step's attention (k_window_attention_step.hip).
#pragma once
#include "device_utils.h"
#include "kernels_stream32.h"

namespace uzu {
namespace k {

// a workgroup per (row, part): the first kGatedKeep coordinates travel in registers, their weights too (every load in front of the sum of squares), wider parts go over
// the rest in further steps
constexpr uint32_t kGatedUnroll = 4, kGatedKeep = 256 * kGatedUnroll;
__device__ __forceinline__ void gated_norm_part(const GatedNormParams& p, uint32_t r, uint32_t part) {
    __shared__ float s_red[16];
    const uint32_t w = p.width / p.parts, c0 = part * w, tid = threadIdx.x;
    const float *y = p.y + (size_t)r * p.ldy + c0, *g = p.gate + (size_t)r * p.ldgate + c0, *wt = p.weight + c0;
    float* out = p.out + (size_t)r * p.ldo + c0;
    auto gated = [](float v, float z) { return v * (z / (1.0f + expf(-z))); };
    float yv[kGatedUnroll], gv[kGatedUnroll], wv[kGatedUnroll], ss = 0.0f;
#pragma unroll
    for (uint32_t u = 0; u < kGatedUnroll; ++u) {
        const uint32_t i = tid + u * 256;
        yv[u] = i < w ? y[i] : 0.0f, gv[u] = i < w ? g[i] : 0.0f, wv[u] = i < w ? wt[i] : 0.0f;
    }
#pragma unroll
    for (uint32_t u = 0; u < kGatedUnroll; ++u) {
        yv[u] = gated(yv[u], gv[u]);
        ss = fmaf(yv[u], yv[u], ss);
    }
    for (uint32_t i = tid + kGatedKeep; i < w; i += 256) {
        const float v = gated(y[i], g[i]);
        ss = fmaf(v, v, ss);
    }
    const float inv = p.out_scale / sqrtf(block_sum(ss, s_red) / (float)w + p.eps);
#pragma unroll
    for (uint32_t u = 0; u < kGatedUnroll; ++u) {
        const uint32_t i = tid + u * 256;
        if (i < w) out[i] = yv[u] * inv * wv[u];
    }
    for (uint32_t i = tid + kGatedKeep; i < w; i += 256) out[i] = gated(y[i], g[i]) * inv * wt[i]; // (out may be y: a thread replaces what it alone reads)
}

} // namespace k
} // namespace uzu
