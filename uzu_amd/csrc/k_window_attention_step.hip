// k_window_attention_step.hip -- attention over cached keys and values (kernels_stream32.h::window_attention) for passes of one row per sequence over bf16 caches: decode steps.
//
// A step's launch is a chain of memory round trips: the sequence's span and cache pointers, then keys and values.  So nothing is staged and nothing else is waited for: L = dim / 8 lanes
// hold a key (16 bytes of it each), 64 / L keys a wave-load, two loads of keys and two of values a wave and turn, all in flight together (the next turn's as well: more registers,
// three workgroups a CU for four, 8 sequences 14 .. 16 us for 12 .. 13).  A workgroup of four waves takes one row's HQ query heads of one key / value head over its share of the row's keys, 1024 / dim keys a turn; scores are exact bf16 x f32 products
// added in f32 over a key's lanes (DPP), the running maximum, sum and weighted values are per group of L lanes, the groups meet at the end: lane swaps that halve the values a lane carries,
// then LDS.  The shares' results leave unnormalised and window_attention_merge adds them; with one share the kernel normalises by itself.
// Beside either launch stand workgroups of other work that a pair of mixers has at the same time: the state-space mixer's recurrence (independent of the attention) and its gated norm
// (independent of the merge).  Each was a launch of its own between two dependent ones.
// Bound by the launch and those round trips.  Us, width 128, window 1024, attention + merge + recurrence + gated norm: one sequence of 8 heads on 2, 16 state heads
// 11.4 + 4.4 + 4.4 + 2.8 (matrix cores; launches apart) -> 6.8 + 3.9; 8 sequences of 16 heads on 4, 32 state heads 14.3 + 3.4 + 6.7 + 3.3 -> 13.0 + 4.0.
#include <algorithm>

#include "decayed_state_steps.h"
#include "device_utils.h"
#include "gated_norm_part.h"
#include "kernels_stream32.h"

namespace uzu {
namespace k {

namespace {

template <int CTRL> __device__ __forceinline__ float dpp_plus(float v) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
// the sum over the L consecutive lanes that contain this one, in every one of them
template <int L> __device__ __forceinline__ float key_sum(float v) {
    v = dpp_plus<0xB1>(v);                         // quad_perm [1, 0, 3, 2]
    v = dpp_plus<0x4E>(v);                         // quad_perm [2, 3, 0, 1]
    if constexpr (L >= 8) v = dpp_plus<0x141>(v);  // row_half_mirror: the other quad of eight
    if constexpr (L >= 16) v = dpp_plus<0x140>(v); // row_mirror: the other eight of the row
    return v;
}
typedef __attribute__((ext_vector_type(2))) uint32_t lane_pair;
// lanes of the lower half of the wave: a's sum over both halves; of the upper half: b's
__device__ __forceinline__ float halves_sum(float a, float b) {
    const lane_pair t = __builtin_bit_cast(lane_pair, __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false));
    return bits_to_f32(t.x) + bits_to_f32(t.y); // (by value: the compiler takes a bit cast of a vector's element for one of its first)
}
// even rows of sixteen lanes: a's sum over this row and the next; odd rows: b's over this row and the one before
__device__ __forceinline__ float rows_sum(float a, float b) {
    const lane_pair t = __builtin_bit_cast(lane_pair, __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false));
    return bits_to_f32(t.x) + bits_to_f32(t.y); // (by value: the compiler takes a bit cast of a vector's element for one of its first)
}

// NB: dim and vdim padded to 32 NB; HQ: query heads of the workgroup.  Workgroup = ((row, block of heads), share), behind them `SIDE`: the workgroups of d's recurrence.
template <int NB, int HQ, bool SIDE>
__global__ void __launch_bounds__(256, 4) window_attention_step_kernel(WindowAttentionParams p, DecayedStateParams d, uint32_t first_side) {
    if (SIDE && blockIdx.x >= first_side) {
        const uint32_t b = blockIdx.x - first_side, n = d.nseq * d.heads;
        decayed_state_steps<8, false>(d, b % n, b / n);
        return;
    }
    constexpr int RP = 32 * NB, L = 4 * NB, KPW = 64 / L, KU = 2, KEYS = 4 * KPW * KU;
    __shared__ float s_o[4][HQ][RP], s_m[4][HQ], s_l[4][HQ];
    const uint32_t hg = p.heads / p.kv_heads, hb = (hg + HQ - 1) / HQ;
    const uint32_t share = blockIdx.x % p.splits, rb = blockIdx.x / p.splits, g = rb / hb % p.kv_heads, h0 = rb % hb * HQ, r = rb / (hb * p.kv_heads); // h0: of the hg heads
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), e0 = lane % L * 8, kl = lane / L;
    const uint32_t t = p.spans[r].start; // (one row per sequence: row r is sequence r's)
    const uint8_t* kc = (const uint8_t*)p.key_caches[r] + ((size_t)g * p.dim + e0) * 2;
    const uint8_t* vc = (const uint8_t*)p.value_caches[r] + ((size_t)g * p.vdim + e0) * 2;
    const uint32_t kpitch = p.kv_heads * p.dim * 2, vpitch = p.kv_heads * p.vdim * 2;
    float q[HQ][8], hscale[HQ];
#pragma unroll
    for (int h = 0; h < HQ; ++h) {
        const uint32_t head = g * hg + min(h0 + h, hg - 1);
        const float* at = p.q + (size_t)r * p.ldq + (size_t)head * p.dim + e0;
        f32x4_v a{0.0f, 0.0f, 0.0f, 0.0f}, b = a;
        if (e0 < p.dim) a = *(const f32x4_v*)at, b = *(const f32x4_v*)(at + 4); // (dim % 8 == 0)
#pragma unroll
        for (int e = 0; e < 4; ++e) q[h][e] = a[e], q[h][4 + e] = b[e];
        hscale[h] = p.head_scale ? p.scale * p.head_scale[head] : p.scale;
    }
    uint32_t lo = (p.window && t + 1 > p.window) ? t + 1 - p.window : 0u;
    if (p.chunk) lo = max(lo, t / p.chunk * p.chunk);
    // this share's keys: whole turns, as equal as turns allow
    const uint32_t n = t - lo + 1, per = (n + p.splits * KEYS - 1) / (p.splits * KEYS) * KEYS, first = lo + share * per, end = min(first + per, t + 1); // (first >= end: none)
    u32x4_v kr[KU], vr[KU];
    auto fetch = [&](uint32_t base, u32x4_v (&kd)[KU], u32x4_v (&vd)[KU]) { // (keys behind the last: zeros)
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            const uint32_t key = base + (wave * KU + u) * KPW + kl;
            kd[u] = vd[u] = u32x4_v{0u, 0u, 0u, 0u};
            if (key < end && e0 < p.dim) kd[u] = *(const u32x4_v*)(kc + (size_t)key * kpitch);
            if (key < end && e0 < p.vdim) vd[u] = *(const u32x4_v*)(vc + (size_t)key * vpitch);
        }
    };
    float m[HQ], l[HQ], o[HQ][8];
#pragma unroll
    for (int h = 0; h < HQ; ++h) {
        m[h] = -1.0e30f, l[h] = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[h][e] = 0.0f;
    }
    for (uint32_t base = first; base < end; base += KEYS) {
        fetch(base, kr, vr);
        float s[KU][HQ];
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            const uint32_t key = base + (wave * KU + u) * KPW + kl;
            float kf[8];
#pragma unroll
            for (int w = 0; w < 4; ++w) kf[2 * w] = bits_to_f32(kr[u][w] << 16), kf[2 * w + 1] = bits_to_f32(kr[u][w] & 0xFFFF0000u);
#pragma unroll
            for (int h = 0; h < HQ; ++h) {
                float dot = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) dot = fmaf(q[h][e], kf[e], dot);
                float sc = key_sum<L>(dot) * hscale[h];
                if (p.soft_cap != 0.0f) { // cap * tanh(s / cap), tanh(x) = 1 - 2 / (1 + e^(2x))
                    const float e2 = fast_exp(2.0f * sc / p.soft_cap);
                    sc = p.soft_cap * (1.0f - 2.0f / (1.0f + e2));
                }
                if (p.dist_bias && key < end) sc += p.dist_bias[(size_t)min(t - key, p.dist_rows - 1) * p.heads + g * hg + min(h0 + h, hg - 1)];
                s[u][h] = key < end ? sc : -INFINITY;
            }
        }
        float vf[KU][8];
#pragma unroll
        for (int u = 0; u < KU; ++u)
#pragma unroll
            for (int w = 0; w < 4; ++w) vf[u][2 * w] = bits_to_f32(vr[u][w] << 16), vf[u][2 * w + 1] = bits_to_f32(vr[u][w] & 0xFFFF0000u);
#pragma unroll
        for (int h = 0; h < HQ; ++h) {
            const float m_new = fmaxf(m[h], fmaxf(s[0][h], s[1][h])), corr = fast_exp(m[h] - m_new), w0 = fast_exp(s[0][h] - m_new), w1 = fast_exp(s[1][h] - m_new); // (masked: 0)
            l[h] = fmaf(l[h], corr, w0 + w1), m[h] = m_new;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[h][e] = fmaf(w1, vf[1][e], fmaf(w0, vf[0][e], o[h][e] * corr));
        }
    }
    // the wave's groups: one maximum, then sums of which each lane keeps two of its eight columns
    const uint32_t own = (lane & 32 ? 4u : 0u) + (lane & 16 ? 2u : 0u);
#pragma unroll
    for (int h = 0; h < HQ; ++h) {
        float mw = m[h];
#pragma unroll
        for (int off = L; off < 64; off <<= 1) mw = fmaxf(mw, __shfl_xor(mw, off, 64));
        const float a = fast_exp(m[h] - mw);
        float lw = l[h] * a;
#pragma unroll
        for (int off = L; off < 64; off <<= 1) lw += __shfl_xor(lw, off, 64);
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = o[h][e] * a;
#pragma unroll
            for (int off = L; off < 16; off <<= 1) v[e] += __shfl_xor(v[e], off, 64);
        }
        float v4[4], v2[2];
#pragma unroll
        for (int e = 0; e < 4; ++e) v4[e] = halves_sum(v[e], v[e + 4]);
#pragma unroll
        for (int e = 0; e < 2; ++e) v2[e] = rows_sum(v4[e], v4[e + 2]);
        if ((lane & 15) < (uint32_t)L) s_o[wave][h][e0 + own] = v2[0], s_o[wave][h][e0 + own + 1] = v2[1];
        if (lane == 0) s_m[wave][h] = mw, s_l[wave][h] = lw;
    }
    lds_barrier();
    for (uint32_t i = tid; i < HQ * RP; i += 256) {
        const uint32_t h = i / RP, c = i % RP;
        if (h0 + h >= hg) break;
        const uint32_t head = g * hg + h0 + h;
        const bool with_sink = p.sinks && share == 0;
        const float sink = with_sink ? p.sinks[head] : -1.0e30f;
        const float top = fmaxf(fmaxf(fmaxf(s_m[0][h], s_m[1][h]), fmaxf(s_m[2][h], s_m[3][h])), sink);
        float acc = 0.0f, den = with_sink ? fast_exp(sink - top) : 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float a = fast_exp(s_m[w][h] - top);
            acc = fmaf(s_o[w][h][c], a, acc), den = fmaf(s_l[w][h], a, den);
        }
        if (p.splits > 1) {
            float* ws = p.split_ws + (((size_t)r * p.heads + head) * p.splits + share) * (RP + 4);
            ws[c] = acc;
            if (c == 0) ws[RP] = top, ws[RP + 1] = den;
        } else if (c < p.vdim) {
            if (p.gate) den *= 1.0f + expf(-p.gate[(size_t)r * p.ldgate + head]);
            p.out[(size_t)r * p.ldo + (size_t)head * p.vdim + c] = acc / den * p.out_scale;
        }
    }
}

// a workgroup per item: out = sum_s e^(m_s - M) O_s / sum_s e^(m_s - M) l_s over the shares (a share that saw no key has l = 0 and m = -1e30); threads 0 .. 127 add the even
// ones, 128 .. 255 the odd ones, both in order, then one to the other.  (gate: the item's result times sigmoid(gate[row, head]), item = row * heads + head.)  Behind the items: the parts of g's norm.
__global__ void __launch_bounds__(256) window_attention_merge_kernel(WindowAttentionParams p, uint32_t rp, GatedNormParams g) {
    const uint32_t items = p.rows * p.heads, tid = threadIdx.x;
    if (blockIdx.x >= items) {
        const uint32_t b = blockIdx.x - items;
        gated_norm_part(g, b / g.parts, b % g.parts);
        return;
    }
    const uint32_t item = blockIdx.x, splits = p.splits, c = tid & 127, odd = tid >> 7, lane = tid & 63;
    const float* base = p.split_ws + (size_t)item * splits * (rp + 4);
    __shared__ float s_w[64], s_half[128];
    // the shares' weights in the first wave, a lane per share (at most 64); its denominator is the same in every lane
    const float m = lane < splits ? base[(size_t)lane * (rp + 4) + rp] : -1.0e30f, l = lane < splits ? base[(size_t)lane * (rp + 4) + rp + 1] : 0.0f;
    const float w = fast_exp(m - wave_max(m));
    float den = wave_sum(w * l);
    if (p.gate) den *= 1.0f + expf(-p.gate[(size_t)(item / p.heads) * p.ldgate + item % p.heads]);
    if (tid < 64) s_w[tid] = w;
    lds_barrier();
    float acc = 0.0f;
    if (c < p.vdim)
#pragma unroll 8
        for (uint32_t s = odd; s < splits; s += 2) acc = fmaf(s_w[s], base[(size_t)s * (rp + 4) + c], acc);
    if (odd) s_half[c] = acc;
    lds_barrier();
    if (!odd && c < p.vdim) p.out[(size_t)(item / p.heads) * p.ldo + (size_t)(item % p.heads) * p.vdim + c] = (acc + s_half[c]) / den * p.out_scale;
}

uint32_t width_blocks(const WindowAttentionParams& p) {
    const uint32_t w = std::max(p.dim, p.vdim);
    return w <= 32 ? 1 : w <= 64 ? 2 : w <= 128 ? 4 : 0;
}
uint32_t heads_a_block(const WindowAttentionParams& p) { return p.heads / p.kv_heads >= 3 ? 4 : p.heads / p.kv_heads; }

} // namespace

bool window_attention_step_supported(const WindowAttentionParams& p) {
    return p.one_row && p.rows == p.nseq && p.cache_bf16 && width_blocks(p) && p.dim % 8 == 0 && p.vdim % 8 == 0 && p.ldq % 4 == 0 && p.kv_heads && p.heads % p.kv_heads == 0 && !p.split_items &&
           ((uintptr_t)p.q & 15) == 0 && (uint64_t)p.kv_heads * 128 * 2 < (1ull << 32) && (p.splits == 1 || (p.splits > 1 && p.splits <= 64 && p.split_ws && p.split_ws_bytes >= window_attention_split_ws_bytes(p.rows, p.heads, p.splits)));
}
// Shares: a turn of keys each, at most 32, and two workgroups a CU in all (8 sequences of 4 key / value heads: 8 / 16 / 32 shares 14.5 / 12.1 .. 13.4 / 14.6 us); up to two turns one
// share, which needs no merge.
uint32_t window_attention_step_splits(const WindowAttentionParams& p, uint32_t keys, uint32_t num_cus) {
    const uint32_t turn = 128 / width_blocks(p), blocks = (keys + turn - 1) / turn, hg = p.heads / p.kv_heads, hq = heads_a_block(p), each = p.rows * p.kv_heads * ((hg + hq - 1) / hq);
    if (blocks <= 2) return 1;
    return std::min(blocks, std::max(1u, std::min(32u, 2 * num_cus / std::max(1u, each))));
}

// Us, with the merge: every share is a workgroup's turns, one behind the other.  (8580 passes of key / value heads with five query heads and more: within 5 % on the average)
float window_attention_step_us(const WindowAttentionParams& p, uint32_t seen) {
    const bool wide = width_blocks(p) > 2;
    const uint32_t turn = 128 / width_blocks(p), hg = p.heads / p.kv_heads, hq = heads_a_block(p), share = turn * p.splits;
    return (wide ? 4.0f : 4.35f) + (wide ? 0.033f : 0.020f) * 1e-3f * (float)seen * (float)(p.rows * p.kv_heads * ((hg + hq - 1) / hq)) + (wide ? 1.21f : 1.06f) * (float)((seen + share - 1) / share) +
           (p.splits > 1 ? 3.7f : 0.0f) + (wide ? 0.43e-3f : 0.27e-3f) * (float)p.rows * (float)(p.heads * p.splits);
}

uzu_status window_attention_step(hipStream_t s, const WindowAttentionParams& p, const DecayedStateParams* beside) {
    UZU_REQUIRE(window_attention_step_supported(p), "window_attention_step: one row per sequence over bf16 caches, with its workspace");
    UZU_REQUIRE(!beside || window_attention_step_beside(*beside), "window_attention_step: a recurrence of one decay per head and up to 128 key channels");
    const uint32_t hg = p.heads / p.kv_heads, hq = heads_a_block(p), nb = width_blocks(p);
    const uint64_t own = (uint64_t)p.rows * p.kv_heads * ((hg + hq - 1) / hq) * p.splits, side = beside ? (uint64_t)beside->nseq * beside->heads * ((beside->vdim + 15) / 16) : 0;
    UZU_REQUIRE(own + side <= 0x7FFFFFFFu, "window_attention_step: too many heads for one launch");
    const DecayedStateParams d = beside ? *beside : DecayedStateParams{};
#define UZU_WS(NB, HQ)                                                                                                                                                                    \
    return launch_check([&] {                                                                                                                                                             \
        if (beside) hipLaunchKernelGGL((window_attention_step_kernel<NB, HQ, true>), dim3((uint32_t)(own + side)), dim3(256), 0, s, p, d, (uint32_t)own);                                 \
        else hipLaunchKernelGGL((window_attention_step_kernel<NB, HQ, false>), dim3((uint32_t)own), dim3(256), 0, s, p, d, (uint32_t)own);                                                \
    }, "window_attention_step")
    if (nb == 1 && hq == 1) UZU_WS(1, 1);
    if (nb == 1 && hq == 2) UZU_WS(1, 2);
    if (nb == 1) UZU_WS(1, 4);
    if (nb == 2 && hq == 1) UZU_WS(2, 1);
    if (nb == 2 && hq == 2) UZU_WS(2, 2);
    if (nb == 2) UZU_WS(2, 4);
    if (hq == 1) UZU_WS(4, 1);
    if (hq == 2) UZU_WS(4, 2);
    UZU_WS(4, 4);
#undef UZU_WS
}
bool window_attention_step_beside(const DecayedStateParams& d) {
    return d.per_head && d.dim >= 1 && d.dim <= 128 && d.rows_in && d.decay && d.out && d.states && d.spans && d.heads && d.groups && d.heads % d.groups == 0 && d.a_log && d.dt_bias && d.nseq && d.rows == d.nseq;
}

uzu_status window_attention_merge(hipStream_t s, const WindowAttentionParams& p, const GatedNormParams* beside) {
    const GatedNormParams g = beside ? *beside : GatedNormParams{};
    UZU_REQUIRE(!beside || (g.y && g.gate && g.weight && g.out && g.width && g.parts && g.width % g.parts == 0), "window_attention_merge: %u coordinates in %u equal parts", g.width, g.parts);
    UZU_REQUIRE(p.splits > 1 && p.splits <= 64 && (uint64_t)p.rows * p.heads + (uint64_t)g.rows * g.parts <= 0x7FFFFFFFu, "window_attention_merge: %u shares", p.splits);
    return launch_check([&] { hipLaunchKernelGGL(window_attention_merge_kernel, dim3(p.rows * p.heads + g.rows * g.parts), dim3(256), 0, s, p, 32 * width_blocks(p), g); }, "window_attention_merge");
}

} // namespace k
} // namespace uzu
