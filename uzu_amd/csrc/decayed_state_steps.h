// decayed_state_steps.h -- the decayed outer-product state walked token by token (k_decayed_state.hip): the body of a launch of its own, and of the workgroups
// that stand beside a decode step's attention (k_window_attention_step.hip).
#pragma once
#include "device_utils.h"
#include "kernels_stream32.h"

namespace uzu {
namespace k {

__device__ __forceinline__ float softplus_f32(float z) { return fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z))); }

// one decay per head: the step size of a row (it multiplies the key); the row's log decay is -exp(a_log) times it
__device__ __forceinline__ float head_step(const DecayedStateParams& p, uint32_t r, uint32_t a) { return softplus_f32(p.decay[(size_t)r * p.lddecay + a] + p.dt_bias[a]); }
// a decay per key channel: sigmoid(z)^inv_temperature by way of its logarithm, min(z, 0) - ln(1 + e^(-|z|)) (an absolute error of one rounding of 1: what the decay
// itself is rounded to)
__device__ __forceinline__ float channel_decay(float z, float inv_temperature) { return fast_exp((fminf(z, 0.0f) - fast_log(1.0f + fast_exp(-fabsf(z)))) * inv_temperature); }

// ---- token by token, a workgroup of 256 per (sequence * heads, block of 16 value columns); thread = (column tid % 16, part tid / 16 of the key channels): it owns S[i][column] for
// i = part, part + 16, ...; a token's partial sums meet by lane exchange and then over the four waves in LDS, in a fixed order
template <int N, bool CHANNEL> // N: channels per thread (dim <= 16 N)
__device__ __forceinline__ void decayed_state_steps(const DecayedStateParams& p, uint32_t seq_head, uint32_t col_block) {
    __shared__ float s_q[16 * N], s_k[16 * N], s_e[CHANNEL ? 16 * N : 1], s_v[16], s_red[4][16];
    const uint32_t z = seq_head / p.heads, a = seq_head % p.heads, g = a / (p.heads / p.groups);
    const uint32_t tid = threadIdx.x, cl = tid & 15, part = tid >> 4, wave = tid >> 6, col = col_block * 16 + cl;
    const SeqSpan sp = p.spans[z];
    if (!sp.count) return;
    const bool live = col < p.vdim;
    float* state = p.states[z] + (size_t)a * p.dim * p.vdim;
    float S[N];
#pragma unroll
    for (int n = 0; n < N; ++n) {
        const uint32_t i = part + 16 * n;
        S[n] = (sp.start && live && i < p.dim) ? state[(size_t)i * p.vdim + col] : 0.0f;
    }
    const float rate = CHANNEL ? 0.0f : expf(p.a_log[a]);
    for (uint32_t t = 0; t < sp.count; ++t) {
        const uint32_t r = sp.row0 + t;
        const float* row = p.rows_in + (size_t)r * p.ld;
        float decay = 0.0f, step = 1.0f;
        if (!CHANNEL) step = head_step(p, r, a), decay = expf(-rate * step);
        for (uint32_t c = tid; c < 16 * N; c += 256) { // (channels beyond dim: zeros, so that the padding rows of S stay zero)
            const bool in = c < p.dim;
            s_q[c] = in ? row[p.q_col + (size_t)g * p.dim + c] * p.q_scale : 0.0f;
            s_k[c] = in ? row[p.k_col + (size_t)g * p.dim + c] * step : 0.0f;
            if (CHANNEL) s_e[c] = in ? channel_decay(p.decay[(size_t)r * p.lddecay + (size_t)a * p.dim + c], p.inv_temperature) : 0.0f;
        }
        if (tid < 16) s_v[tid] = live ? row[p.v_col + (size_t)a * p.vdim + col] : 0.0f;
        __syncthreads();
        const float v = s_v[cl];
        float sum = 0.0f;
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const uint32_t i = part + 16 * n;
            S[n] = fmaf(CHANNEL ? s_e[i] : decay, S[n], s_k[i] * v);
            sum = fmaf(S[n], s_q[i], sum);
        }
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        if ((tid & 63) < 16) s_red[wave][cl] = sum;
        __syncthreads();
        if (tid < 16 && live) {
            float o = (s_red[0][cl] + s_red[1][cl]) + (s_red[2][cl] + s_red[3][cl]);
            if (p.skip) o = fmaf(p.skip[a], v, o);
            p.out[((size_t)r * p.heads + a) * p.vdim + col] = o;
        }
    }
    if (!live) return;
#pragma unroll
    for (int n = 0; n < N; ++n) {
        const uint32_t i = part + 16 * n;
        if (i < p.dim) state[(size_t)i * p.vdim + col] = S[n];
    }
}

} // namespace k
} // namespace uzu
