// k_step32.hip -- launches of an f32-stream design's decode step that do the work of several (kernels_stream32.h): a pass of a few rows is a chain of launches of 3 to 7 us whose bodies
// are memory round trips, so what only one row's workgroup would do is done in front of (or by every workgroup of) the launch that reads it.
// Us, width 1024, 2 of 8 experts of 1024: rms_norm_add_rows 3.1 + moe_route_groups 5.0 + moe_experts_gate_up 6.8 -> norm_route_gate_up 7.4 (256 workgroups that each read 36 KB of the
// same numbers from the L2, 8 KB of experts' rows a wave); 8 rows of 2048: 4.3 + 7.0 -> norm_route_rows 5.5.  rms_norm_add_rows 3.1 + a projection onto 4112 columns 4.7 -> norm_linear 6.9;
// ... + rms_norm_rows 2.8 + the read-out onto 32768 15.6 + argmax_pass1 4.7 -> 14.9; argmax_pass2 4.3 + commit 2.9 + embed_rows 3.8 + rms_norm_rows 2.8 -> step_turn 4.2.
#include <algorithm>

#include "device_utils.h"
#include "kernels_stream32.h"
#include "stream32_epilogue.h"

namespace uzu {
namespace k {

namespace {

constexpr uint32_t kStepThreads = 512, kStepWaves = kStepThreads / 64, kStepUnroll = 2, kStepMaxWidth = 4 * kStepThreads * kStepUnroll; // 4096 coordinates, four neighbours a thread
constexpr uint32_t kStepMaxOutputs = 64, kStepMaxTop = 8;

__device__ __forceinline__ float step_operand(float v, uint32_t bf16_products) { return bf16_products ? round_bf16(v) : v; }

// the order of arg-max candidates (k_elementwise.hip): the larger value, of equal ones the lower index; a NaN never wins
__device__ __forceinline__ void step_amax(float& bv, uint32_t& bi, float v, uint32_t i) {
    if (v > bv || (v == bv && i < bi)) bv = v, bi = i;
}
// over the workgroup; the result in thread 0
__device__ __forceinline__ void step_amax_block(float& bv, uint32_t& bi, float* s_v, uint32_t* s_i) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off, 64);
        const uint32_t oi = __shfl_xor(bi, off, 64);
        step_amax(bv, bi, ov, oi);
    }
    if ((threadIdx.x & 63) == 0) s_v[threadIdx.x >> 6] = bv, s_i[threadIdx.x >> 6] = bi;
    __syncthreads();
    if (threadIdx.x == 0)
        for (uint32_t w = 1; w < kStepWaves; ++w) step_amax(bv, bi, s_v[w], s_i[w]);
}

// A row's stream: new = residual + rms(y) * (scales + offset) * layer_scale, its norm for the sublayer that follows left in s_x (rounded if it enters bf16 products).  `write`: the
// row and its norm go to memory as well.  Everything is loaded before the first sum is known.
__device__ __forceinline__ void step_norm_add(const NormAddParams& p, uint32_t r, float* s_x, float* s_red, uint32_t bf16_products, bool write) {
    const uint32_t tid = threadIdx.x, d = p.d;
    f32x4_v yv[kStepUnroll], rv[kStepUnroll], sv[kStepUnroll], lv[kStepUnroll], nv[kStepUnroll];
    float acc = 0.0f, acc2 = 0.0f;
#pragma unroll
    for (uint32_t u = 0; u < kStepUnroll; ++u) {
        const uint32_t i = (tid + u * kStepThreads) * 4;
        yv[u] = rv[u] = sv[u] = nv[u] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f}, lv[u] = f32x4_v{1.0f, 1.0f, 1.0f, 1.0f};
        if (i >= d) continue;
        yv[u] = *(const f32x4_v*)(p.y + (size_t)r * d + i), rv[u] = *(const f32x4_v*)(p.residual + (size_t)r * d + i), sv[u] = *(const f32x4_v*)(p.scales + i);
        nv[u] = *(const f32x4_v*)(p.next_scales + i);
        if (p.layer_scale) lv[u] = *(const f32x4_v*)(p.layer_scale + i);
    }
#pragma unroll
    for (uint32_t u = 0; u < kStepUnroll; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = fmaf(yv[u][e], yv[u][e], acc);
    const float inv = 1.0f / sqrtf(block_sum(acc, s_red) / (float)d + p.eps);
#pragma unroll
    for (uint32_t u = 0; u < kStepUnroll; ++u) {
        const bool in = (tid + u * kStepThreads) * 4 < d;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float v = yv[u][e] * inv * (sv[u][e] + p.offset);
            if (p.layer_scale) v *= lv[u][e];
            rv[u][e] = rv[u][e] + v;
            if (in) acc2 = fmaf(rv[u][e], rv[u][e], acc2);
        }
    }
    const float inv2 = 1.0f / sqrtf(block_sum(acc2, s_red) / (float)d + p.next_eps);
#pragma unroll
    for (uint32_t u = 0; u < kStepUnroll; ++u) {
        const uint32_t i = (tid + u * kStepThreads) * 4;
        if (i >= d) continue;
        f32x4_v x, op;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = rv[u][e] * inv2 * (nv[u][e] + p.next_offset), op[e] = step_operand(x[e], bf16_products);
        *(f32x4_v*)(s_x + i) = op;
        if (write) *(f32x4_v*)(p.out + (size_t)r * d + i) = rv[u], *(f32x4_v*)(p.next + (size_t)r * d + i) = x;
    }
}

// The row's winners (moe_route_groups without a choice of groups): a wave per output, then every wave ranks the outputs, a lane each.  w: the router row of this wave's first output,
// loaded before the row was known.
struct StepChoice {
    int32_t id[kStepMaxTop];
    float weight[kStepMaxTop];
};
__device__ __forceinline__ void step_router_row(const RouteGroupsParams& p, uint32_t e, uint32_t lane, u32x4_v (&w)[kStepMaxWidth / 512]) {
#pragma unroll
    for (uint32_t j = 0; j < kStepMaxWidth / 512; ++j)
        if (j * 512 + lane * 8 < p.d) w[j] = *(const u32x4_v*)(p.router + (size_t)e * p.d + j * 512 + lane * 8);
}
template <uint32_t TOP> __device__ __forceinline__ void step_choose(const RouteGroupsParams& p, const float* s_x, float* s_score, u32x4_v (&w)[kStepMaxWidth / 512], StepChoice& c) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (uint32_t e = wave; e < p.outputs; e += kStepWaves) {
        if (e != wave) step_router_row(p, e, lane, w);
        float z = 0.0f;
#pragma unroll
        for (uint32_t j = 0; j < kStepMaxWidth / 512; ++j) {
            const uint32_t k0 = j * 512 + lane * 8;
            if (k0 >= p.d) break;
            const f32x4_v a = *(const f32x4_v*)(s_x + k0), b = *(const f32x4_v*)(s_x + k0 + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                z = fmaf(i < 2 ? a[2 * i] : b[2 * i - 4], bits_to_f32(w[j][i] << 16), z);
                z = fmaf(i < 2 ? a[2 * i + 1] : b[2 * i - 3], bits_to_f32(w[j][i] & 0xFFFF0000u), z);
            }
        }
        const float sc = 1.0f / (1.0f + expf(-wave_sum(z)));
        if (lane == 0) s_score[e] = sc;
    }
    __syncthreads();
    // an output's rank: how many stand above it (a larger choice score; an equal one of a lower index).  What is not above -infinity (a NaN too) has none and is never chosen.
    const bool in = lane < p.outputs;
    const float mine = in ? s_score[lane] + (p.selection_bias ? p.selection_bias[lane] : 0.0f) : -INFINITY;
    const bool ranked = in && mine > -INFINITY;
    uint32_t rank = 0;
    for (uint32_t o = 0; o < p.outputs; ++o) {
        const float other = bits_to_f32(__builtin_amdgcn_readlane(f32_to_bits(mine), o));
        rank += (other > mine || (other == mine && o < lane)) ? 1u : 0u;
    }
    float sum = 0.0f;
#pragma unroll
    for (uint32_t t = 0; t < TOP; ++t) {
        if (t >= p.top) break;
        const unsigned long long who = __ballot(ranked && rank == t);
        c.id[t] = who ? (int32_t)__builtin_ctzll(who) : -1; // (a row of NaNs has no winner)
        c.weight[t] = who ? s_score[c.id[t]] : 0.0f;
        sum += c.weight[t];
    }
#pragma unroll
    for (uint32_t t = 0; t < TOP; ++t) {
        if (t >= p.top) break;
        c.weight[t] = (p.raw ? c.weight[t] : c.weight[t] / (sum + 1e-20f)) * p.scale;
    }
}

// a workgroup per row: the row joins the stream, is normed and routed
__global__ void __launch_bounds__(kStepThreads) norm_route_rows_kernel(NormAddParams n, RouteGroupsParams p) {
    extern __shared__ __attribute__((aligned(16))) float s_x[]; // [d]
    __shared__ float s_red[16], s_score[kStepMaxOutputs];
    const uint32_t r = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u32x4_v w[kStepMaxWidth / 512] = {};
    if (wave < p.outputs) step_router_row(p, wave, lane, w);
    step_norm_add(n, r, s_x, s_red, p.bf16_products, true);
    __syncthreads();
    StepChoice c;
    step_choose<kStepMaxTop>(p, s_x, s_score, w, c);
    if (threadIdx.x != 0) return;
#pragma unroll
    for (uint32_t t = 0; t < kStepMaxTop; ++t)
        if (t < p.top) p.ids[(size_t)r * p.top + t] = c.id[t], p.weights[(size_t)r * p.top + t] = c.weight[t];
}

// One row: every workgroup norms and routes it for itself, then a wave per hidden unit of a winner (gate and up rows together); the first workgroup writes what later launches read.
__global__ void __launch_bounds__(kStepThreads) norm_route_gate_up_kernel(NormAddParams n, RouteGroupsParams p, const uint16_t* w13, float* hidden, uint32_t ff, ExpertAct act, uint32_t weight_on_input) {
    extern __shared__ __attribute__((aligned(16))) float s_x[]; // [d]
    __shared__ float s_red[16], s_score[kStepMaxOutputs];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), d = p.d;
    u32x4_v w[kStepMaxWidth / 512] = {};
    if (wave < p.outputs) step_router_row(p, wave, lane, w);
    step_norm_add(n, 0, s_x, s_red, p.bf16_products, blockIdx.x == 0);
    __syncthreads();
    StepChoice c;
    step_choose<kStepMaxTop>(p, s_x, s_score, w, c);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
#pragma unroll
        for (uint32_t t = 0; t < kStepMaxTop; ++t)
            if (t < p.top) p.ids[t] = c.id[t], p.weights[t] = c.weight[t];
    }
    for (uint32_t i = blockIdx.x * kStepWaves + wave; i < p.top * ff; i += gridDim.x * kStepWaves) {
        const uint32_t slot = i / ff, f = i - slot * ff;
        int32_t e = -1;
        float wt = 1.0f;
#pragma unroll
        for (uint32_t t = 0; t < kStepMaxTop; ++t)
            if (t == slot) e = c.id[t], wt = weight_on_input ? c.weight[t] : 1.0f;
        if (e < 0) continue;
        const uint16_t* wu = w13 + ((size_t)e * 2 * ff + f) * d;
        const uint16_t* wg = wu + (size_t)ff * d;
        float au = 0.0f, ag = 0.0f;
#pragma unroll 4
        for (uint32_t k0 = lane * 8; k0 < d; k0 += 512) {
            const u32x4_v uv = *(const u32x4_v*)(wu + k0), gv = *(const u32x4_v*)(wg + k0);
            const f32x4_v a = *(const f32x4_v*)(s_x + k0), b = *(const f32x4_v*)(s_x + k0 + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float x0 = j < 2 ? a[2 * j] : b[2 * j - 4], x1 = j < 2 ? a[2 * j + 1] : b[2 * j - 3];
                au = fmaf(x0, bits_to_f32(uv[j] << 16), au), au = fmaf(x1, bits_to_f32(uv[j] & 0xFFFF0000u), au);
                ag = fmaf(x0, bits_to_f32(gv[j] << 16), ag), ag = fmaf(x1, bits_to_f32(gv[j] & 0xFFFF0000u), ag);
            }
        }
        au = wave_sum(au), ag = wave_sum(ag);
        if (lane == 0) hidden[(size_t)slot * ff + f] = expert_act(wt * ag, wt * au, act);
    }
}

// One row: every workgroup norms it for itself, then a wave per output column and turn, the next column's weights on their way; J: pieces of 512 of a row.  AMAX: a workgroup's largest value
// and its column as well (the read-out).
template <int J, bool AMAX>
__global__ void __launch_bounds__(kStepThreads) norm_linear_kernel(NormAddParams n, LinearF32Params p, float* part_value, uint32_t* part_index) {
    extern __shared__ __attribute__((aligned(16))) float s_x[]; // [k]
    __shared__ float s_red[16];
    __shared__ uint32_t s_i[kStepWaves];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = gridDim.x * kStepWaves, k = p.k;
    u32x4_v w[J], next[J];
    auto load = [&](uint32_t col, u32x4_v (&to)[J]) {
        const uint16_t* row = p.w + (size_t)min(col, p.n - 1) * k;
#pragma unroll
        for (int j = 0; j < J; ++j) to[j] = *(const u32x4_v*)(row + min(j * 512 + lane * 8, k - 8)); // (the last piece may pass the row's end: `in_last`)
    };
    uint32_t col = blockIdx.x * kStepWaves + wave;
    const bool in_last = (J - 1) * 512 + lane * 8 < k;
    load(col, w);
    step_norm_add(n, 0, s_x, s_red, p.bf16_products, blockIdx.x == 0);
    __syncthreads();
    float x[J][8];
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) x[j][e] = j * 512 + lane * 8 < k ? s_x[j * 512 + lane * 8 + e] : 0.0f;
    float bv = -INFINITY;
    uint32_t bi = 0xFFFFFFFFu;
    for (; col < p.n; col += waves) {
        load(col + waves, next);
#pragma unroll
        for (int i = 0; i < 4; ++i) w[J - 1][i] = in_last ? w[J - 1][i] : 0u; // (a zero coordinate does not stand against a weight that is not finite)
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc = fmaf(x[j][2 * i], bits_to_f32(w[j][i] << 16), acc);
                acc = fmaf(x[j][2 * i + 1], bits_to_f32(w[j][i] & 0xFFFF0000u), acc);
            }
        acc = wave_sum(acc);
        const float v = linear_epilogue(acc, p.bias ? bf16_to_f32(p.bias[col]) : 0.0f, p, 0, 0, col);
        if (lane == 0) p.y[col] = v;
        if (AMAX) step_amax(bv, bi, col == 0 && !(v == v) ? INFINITY : v, col); // (a NaN in front is never replaced)
#pragma unroll
        for (int j = 0; j < J; ++j) w[j] = next[j];
    }
    if (!AMAX) return;
    step_amax_block(bv, bi, s_red, s_i);
    if (threadIdx.x == 0) part_value[blockIdx.x] = bv, part_index[blockIdx.x] = bi;
}

// What stands between the read-out of a decode step and the first projection of the next one: the choice among the parts' largest logits, the sequence's control block moved on, the chosen token's
// embedding row and its norm.
__global__ void __launch_bounds__(kStepThreads) step_turn_kernel(StepTurnParams p) {
    __shared__ float s_red[16];
    __shared__ uint32_t s_i[kStepWaves + 1];
    const uint32_t tid = threadIdx.x;
    float sv[kStepUnroll][4];
#pragma unroll
    for (uint32_t u = 0; u < kStepUnroll; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) sv[u][e] = (p.normed && (tid + u * kStepThreads) * 4 < p.d) ? p.scales[(tid + u * kStepThreads) * 4 + e] : 0.0f;
    if (p.parts) {
        const uint32_t len = *p.ctx_len;
        float bv = -INFINITY;
        uint32_t bi = 0xFFFFFFFFu;
        for (uint32_t i = tid; i < p.parts; i += kStepThreads) step_amax(bv, bi, p.part_value[i], p.part_index[i]);
        step_amax_block(bv, bi, s_red, s_i);
        if (tid == 0) {
            if (bi == 0xFFFFFFFFu) bi = 0;
            s_i[kStepWaves] = bi;
            *p.out_token = bi, p.sampled[len] = bi, p.tokens[0] = bi, *p.ctx_len = len + 1, p.span->start = len + 1;
        }
    } else if (tid == 0) s_i[kStepWaves] = p.tokens[0]; // (in front of the first step)
    __syncthreads();
    uint32_t t = s_i[kStepWaves];
    if (t >= p.vocab) t = 0;
    f32x4_v x[kStepUnroll];
    float acc = 0.0f;
#pragma unroll
    for (uint32_t u = 0; u < kStepUnroll; ++u) {
        const uint32_t i = (tid + u * kStepThreads) * 4;
        x[u] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
        if (i >= p.d) continue;
        const u32x2_v b = *(const u32x2_v*)(p.table + (size_t)t * p.d + i);
        x[u] = f32x4_v{bits_to_f32(b.x << 16), bits_to_f32(b.x & 0xFFFF0000u), bits_to_f32(b.y << 16), bits_to_f32(b.y & 0xFFFF0000u)};
#pragma unroll
        for (int e = 0; e < 4; ++e) x[u][e] *= p.scale, acc = fmaf(x[u][e], x[u][e], acc);
        *(f32x4_v*)(p.out + i) = x[u];
    }
    if (!p.normed) return;
    const float inv = 1.0f / sqrtf(block_sum(acc, s_red) / (float)p.d + p.eps);
#pragma unroll
    for (uint32_t u = 0; u < kStepUnroll; ++u) {
        const uint32_t i = (tid + u * kStepThreads) * 4;
        if (i >= p.d) continue;
        f32x4_v o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = x[u][e] * inv * (sv[u][e] + p.offset);
        *(f32x4_v*)(p.normed + i) = o;
    }
}

// as many columns a wave as 512 workgroups need, and no more workgroups than those columns take (each reads the row and its weights for itself)
uint32_t norm_linear_blocks(uint32_t n) {
    const uint32_t each = (n + kStepWaves * kNormLinearParts - 1) / (kStepWaves * kNormLinearParts) * kStepWaves;
    return (n + each - 1) / each;
}

} // namespace

// One workgroup writes the row's new stream and norm, and all of them their results, while others may still read the old stream and the sublayer's result
static bool apart_from_row(const NormAddParams& n, const float* written, size_t count) {
    const auto apart = [&](const float* read) { return (uintptr_t)(written + count) <= (uintptr_t)read || (uintptr_t)(read + n.d) <= (uintptr_t)written; };
    return apart(n.y) && apart(n.residual);
}
bool norm_linear_supported(const NormAddParams& n, const LinearF32Params& p) {
    return n.rows == 1 && p.rows == 1 && p.batch == 1 && norm_add_step_supported(n) && apart_from_row(n, n.out, n.d) && apart_from_row(n, n.next, n.d) && apart_from_row(n, p.y, p.n) && p.k == n.d && p.n && p.y && p.w && ((uintptr_t)p.w & 15) == 0 && !p.residual &&
           !p.gate && !p.mul_table && !p.row_offsets && !p.row_map;
}
uzu_status norm_linear(hipStream_t s, const NormAddParams& n, const LinearF32Params& p, float* part_value, uint32_t* part_index, uint32_t* parts) {
    UZU_REQUIRE(norm_linear_supported(n, p) && (!part_value) == (!part_index), "norm_linear: one row of %u (a multiple of 8, up to %u)", n.d, kStepMaxWidth);
    const dim3 grid(norm_linear_blocks(p.n));
    if (parts) *parts = grid.x;
#define UZU_NL(J)                                                                                                                                                                \
    return launch_check([&] {                                                                                                                                                    \
        if (part_value) hipLaunchKernelGGL((norm_linear_kernel<J, true>), grid, dim3(kStepThreads), (size_t)n.d * 4, s, n, p, part_value, part_index);                           \
        else hipLaunchKernelGGL((norm_linear_kernel<J, false>), grid, dim3(kStepThreads), (size_t)n.d * 4, s, n, p, part_value, part_index);                                     \
    }, "norm_linear")
    switch ((n.d + 511) / 512) { // (a piece that lies past the row's end is loaded for nothing: 2560 with eight, 4096 columns 14.4 us; with five 11.7)
    case 1: UZU_NL(1);
    case 2: UZU_NL(2);
    case 3: UZU_NL(3);
    case 4: UZU_NL(4);
    case 5: UZU_NL(5);
    case 6: UZU_NL(6);
    case 7: UZU_NL(7);
    default: UZU_NL(8);
    }
#undef UZU_NL
}
bool step_turn_supported(const StepTurnParams& p) {
    return p.d >= 8 && p.d % 8 == 0 && p.d <= kStepMaxWidth && p.table && p.out && p.tokens && (((uintptr_t)p.table | (uintptr_t)p.out | (uintptr_t)p.normed) & 15) == 0 && (!p.normed || p.scales);
}
uzu_status step_turn(hipStream_t s, const StepTurnParams& p) {
    UZU_REQUIRE(step_turn_supported(p) && (!p.parts || (p.part_value && p.part_index && p.ctx_len && p.out_token && p.sampled && p.span)), "step_turn: rows of %u", p.d);
    return launch_check([&] { hipLaunchKernelGGL(step_turn_kernel, dim3(1), dim3(kStepThreads), 0, s, p); }, "step_turn");
}

bool norm_add_step_supported(const NormAddParams& n) {
    return n.d >= 8 && n.d % 8 == 0 && n.d <= kStepMaxWidth && n.y && n.residual && n.out && n.scales && n.next && n.next_scales &&
           (((uintptr_t)n.y | (uintptr_t)n.residual | (uintptr_t)n.out | (uintptr_t)n.scales | (uintptr_t)n.layer_scale | (uintptr_t)n.next | (uintptr_t)n.next_scales) & 15) == 0;
}
bool norm_route_supported(const NormAddParams& n, const RouteGroupsParams& p) {
    return norm_add_step_supported(n) && p.d == n.d && n.rows == p.rows && p.keep == p.groups && p.outputs >= 1 && p.outputs <= kStepMaxOutputs && p.top >= 1 && p.top <= std::min(p.outputs, kStepMaxTop) &&
           p.router && p.ids && p.weights && ((uintptr_t)p.router & 15) == 0;
}
// Eight waves have a workgroup's outputs here, sixteen in moe_route_groups: of many outputs of short rows, whose row is no work, the second is as much faster as a launch costs.  Us, apart and joined (with the
// experts behind): 64 outputs, 8 rows of 256 15.3 / 16.2, 1024 22.0 / 22.1, 2048 43.3 / 41.1, 64 rows of 512 31.0 / 31.9; 32 outputs, 8 rows of 1024 25.5 / 23.5.  With the first products in the same launch it
// is the faster one at every size that it takes, though every workgroup works the choice out for itself: one row, 2 winners of 1024, 64 outputs of 256 11.6 / 10.9 (512 hidden units), of 1024 18.2 / 13.5, of 2048
// 21.9 / 14.8, of 4096 54.3 / 24.0; 8 winners of 64, 4096 83.1 / 41.5.
bool norm_route_faster(const RouteGroupsParams& p) { return p.outputs <= 32 || p.d >= 1536; }
uzu_status norm_route_rows(hipStream_t s, const NormAddParams& n, const RouteGroupsParams& p) {
    if (!p.rows) return UZU_OK;
    UZU_REQUIRE(norm_route_supported(n, p), "norm_route: rows of %u, %u of %u outputs", n.d, p.top, p.outputs);
    return launch_check([&] { hipLaunchKernelGGL(norm_route_rows_kernel, dim3(p.rows), dim3(kStepThreads), (size_t)p.d * 4, s, n, p); }, "norm_route_rows");
}
bool norm_route_gate_up_supported(const NormAddParams& n, const RouteGroupsParams& p, const uint16_t* w13, uint32_t ff, const ExpertAct& act) {
    return p.rows == 1 && norm_route_supported(n, p) && apart_from_row(n, n.out, n.d) && apart_from_row(n, n.next, n.d) && !act.plain && ff >= 1 && ((uintptr_t)w13 & 15) == 0;
}
uzu_status norm_route_gate_up(hipStream_t s, const NormAddParams& n, const RouteGroupsParams& p, const uint16_t* w13, float* hidden, uint32_t ff, const ExpertAct& act, uint32_t weight_on_input) {
    UZU_REQUIRE(w13 && hidden && norm_route_gate_up_supported(n, p, w13, ff, act) && apart_from_row(n, hidden, (size_t)p.top * ff),
                "norm_route_gate_up: one row, gated experts, what is written apart from the old row and what joins it");
    const uint32_t blocks = std::min((p.top * ff + kStepWaves - 1) / kStepWaves, 512u);
    return launch_check([&] { hipLaunchKernelGGL(norm_route_gate_up_kernel, dim3(blocks), dim3(kStepThreads), (size_t)p.d * 4, s, n, p, w13, hidden, ff, act, weight_on_input); }, "norm_route_gate_up");
}

} // namespace k
} // namespace uzu
