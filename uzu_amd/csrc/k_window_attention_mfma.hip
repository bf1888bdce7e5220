// k_window_attention_mfma.hip -- the matrix-core form of the attention over cached keys and values (kernels_stream32.h::window_attention): prompt-sized
// passes over bf16 caches.
//
// Items are (row, query head) pairs of ONE sequence and ONE key / value head: a wave owns 32 of them, a workgroup of a prompt 128, so with heads / kv_heads = 4 a
// workgroup's 32 neighbouring rows share every staged stretch of keys.  Both products are computed transposed with v_mfma_f32_32x32x16_bf16, so that a lane
// owns one item:
//   S^T = K Q^T     A = the key block [32][dim] from LDS, B = the item's query, rounded to bf16 as hi + lo (two products: the query keeps 16 significant bits);
//                   the result gives a lane 16 key scores of ITS item, so scale, cap, mask and the running maximum / sum are per-lane work (one exchange
//                   with lane ^ 32);
//   O^T += V^T P^T  A = the value block transposed [vdim][32] from LDS, B = those 16 weights as hi + lo bf16; rescaling and the final 1 / l are per lane.
// The k order inside an MFMA only has to agree between A and B: for O^T the lane's keys are taken in the order the S^T result already holds them.
// Scores, weights and sums are f32; the sink enters as the initial maximum with weight 1 in the denominator.
#include <algorithm>

#include "device_utils.h"
#include "gemm_convert.h"
#include "kernels_stream32.h"

namespace uzu {
namespace k {

namespace {

__device__ __forceinline__ void split_bf16(float a, float b, uint32_t& hi, uint32_t& lo) {
    const uint16_t h0 = f32_to_bf16(a), h1 = f32_to_bf16(b);
    const uint16_t l0 = f32_to_bf16(a - bf16_to_f32(h0)), l1 = f32_to_bf16(b - bf16_to_f32(h1));
    hi = (uint32_t)h0 | ((uint32_t)h1 << 16), lo = (uint32_t)l0 | ((uint32_t)l1 << 16);
}

// IW waves of a workgroup own 32 items each, KG groups of such waves share the keys of a staged stretch (32 KG keys: group i takes its 32), so a workgroup is IW KG waves and
// their unnormalised results meet in LDS at the end, in group order.  Prompts: IW 4, KG 2 (1 where the tiles are many: window_attention_mfma); a pass's tiles are about a workgroup per CU, and a wave alone on its SIMD waits for
// itself at every exponential and every staged block (the next block's loads are in flight meanwhile; values are transposed two keys at a time).  2048 rows of 16 heads on 4,
// width 128, window 1024: 147 us with four waves and no look-ahead, 61 so.  SPLIT (few items, many keys: passes of a few rows a sequence, which k_window_attention_step.hip does not take): grid.z
// workgroups share an item tile's stretches (stretch i goes to workgroup i mod grid.z) and leave unnormalised sums with their running maximum / denominator in p.split_ws;
// window_attention_mfma_merge_kernel combines them.  Two forms (window_attention_split_keys): IW 4, KG 1, stretches of 32 keys, and IW 1, KG 4, stretches of 128 (with IW 4 three waves
// of four have no items, but they help staging).  The sink belongs to group 0 of split 0.
// AHEAD: the next stretch's loads are in flight while one is computed.
template <int NB, int IW, int KG, bool SPLIT, bool AHEAD> // dim and vdim padded to RP = 32 NB
__global__ void __launch_bounds__(64 * IW * KG) window_attention_mfma_kernel(WindowAttentionParams p) {
    constexpr int RP = 32 * NB, KP = RP * 2 + 16, TP = 80, VEC = RP / 8, T = 64 * IW * KG, KEYS = 32 * KG;
    constexpr int KN = (KEYS * VEC + T - 1) / T, VN = (KEYS / 2 * VEC + T - 1) / T; // 16-byte pieces of the keys / pairs of them of the values per thread
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t* s_k = smem;              // [KEYS][KP bytes]
    uint8_t* s_vt = smem + KEYS * KP; // [KG][RP][TP bytes]: 32 keys + pad
    const uint32_t hg = p.heads / p.kv_heads, g = blockIdx.y;
    // the sequence of this tile (tiles of ITEMS items): a lane per sequence, 64 at a time
    constexpr uint32_t ITEMS = 32 * IW;
    uint32_t wg = blockIdx.x, z = p.nseq == 1 ? 0u : 0xFFFFFFFFu, before = 0;
    for (uint32_t z0 = 0; z0 < p.nseq && z == 0xFFFFFFFFu; z0 += 64) {
        const uint32_t ln = threadIdx.x & 63;
        uint32_t upto = z0 + ln < p.nseq ? (p.spans[z0 + ln].count * hg + ITEMS - 1) / ITEMS : 0u;
        for (uint32_t o = 1; o < 64; o <<= 1) {
            const uint32_t below = __shfl_up(upto, o, 64);
            if (ln >= o) upto += below;
        }
        const unsigned long long behind = __ballot(before + upto > wg);
        const uint32_t i = behind ? (uint32_t)__builtin_ctzll(behind) : 64u;
        before += i ? (uint32_t)__builtin_amdgcn_readlane((int)upto, (int)i - 1) : 0u;
        if (behind) z = z0 + i;
    }
    if (z == 0xFFFFFFFFu) return;
    wg -= before;
    const SeqSpan sp = p.spans[z];
    const uint32_t tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6) % IW, kg = __builtin_amdgcn_readfirstlane(tid >> 6) / IW; // (item block, key group)
    const uint32_t items = sp.count * hg;
    auto row_lo = [&](uint32_t t) { // the first key the row at position t sees: the window's edge or its chunk's start, whichever is later
        uint32_t lo = (p.window && t + 1 > p.window) ? t + 1 - p.window : 0u;
        if (p.chunk) lo = max(lo, t / p.chunk * p.chunk);
        return lo;
    };
    // this lane's item
    const uint32_t it = wg * ITEMS + wave * 32 + l32;
    const bool valid = it < items;
    const uint32_t gi = valid ? it : items - 1;
    const uint32_t row = gi / hg, head = g * hg + gi % hg;
    const uint32_t t = sp.start + row, lo = row_lo(t);
    // key ranges of the workgroup and of this wave
    const uint32_t g_last = (wg * ITEMS + ITEMS < items ? wg * ITEMS + ITEMS : items) - 1;
    const uint32_t kmin = row_lo(sp.start + wg * ITEMS / hg), kmax = sp.start + g_last / hg;
    const uint32_t w_first = wg * ITEMS + wave * 32;
    const bool wave_on = w_first < items;
    const uint32_t w_last = (w_first + 32 < items ? w_first + 32 : items) - 1;
    const uint32_t wave_lo = wave_on ? row_lo(sp.start + w_first / hg) : 0, wave_hi = wave_on ? sp.start + w_last / hg : 0;

    u32x4_t qh[2 * NB], ql[2 * NB];
    {
        const float* qrow = p.q + (size_t)(sp.row0 + row) * p.ldq + (size_t)head * p.dim;
#pragma unroll
        for (int s = 0; s < 2 * NB; ++s) {
            const uint32_t k0 = s * 16 + half * 8;
            u32x4_t fh{0u, 0u, 0u, 0u}, fl{0u, 0u, 0u, 0u};
            if (valid && k0 < p.dim) { // dim % 8 == 0: a fragment is inside the head or outside it
                const f32x4_v a = *(const f32x4_v*)(qrow + k0), b = *(const f32x4_v*)(qrow + k0 + 4);
                uint32_t h[4], w[4];
                split_bf16(a.x, a.y, h[0], w[0]), split_bf16(a.z, a.w, h[1], w[1]), split_bf16(b.x, b.y, h[2], w[2]), split_bf16(b.z, b.w, h[3], w[3]);
                fh = u32x4_t{h[0], h[1], h[2], h[3]}, fl = u32x4_t{w[0], w[1], w[2], w[3]};
            }
            qh[s] = fh, ql[s] = fl;
        }
    }
    const bool with_sink = p.sinks && kg == 0 && (!SPLIT || blockIdx.z == 0);
    float m_run = with_sink ? p.sinks[head] : -1.0e30f;
    float l_run = with_sink ? 1.0f : 0.0f;
    f32x16_t o[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[b][r] = 0.0f;
    const uint8_t* kc = (const uint8_t*)p.key_caches[z];
    const uint8_t* vc = (const uint8_t*)p.value_caches[z];
    const size_t kpitch = (size_t)p.kv_heads * p.dim, vpitch = (size_t)p.kv_heads * p.vdim;
    const float inv_cap = p.soft_cap != 0.0f ? 1.0f / p.soft_cap : 0.0f;
    const float hscale = p.head_scale ? p.scale * p.head_scale[head] : p.scale;

    u32x4_v kr[KN], vr[VN][2];
    auto fetch = [&](uint32_t base) { // (keys behind the last: zeros)
#pragma unroll
        for (int i = 0; i < KN; ++i) {
            const uint32_t v = tid + i * T, kk = base + v / VEC, e0 = v % VEC * 8;
            kr[i] = u32x4_v{0u, 0u, 0u, 0u};
            if (v < KEYS * VEC && kk <= kmax && e0 < p.dim) kr[i] = *(const u32x4_v*)(kc + ((size_t)kk * kpitch + (size_t)g * p.dim + e0) * 2);
        }
#pragma unroll
        for (int i = 0; i < VN; ++i) {
            const uint32_t v = tid + i * T, e0 = v / 16 % VEC * 8;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t kk = base + v / (16 * VEC) * 32 + v % 16 * 2 + j;
                vr[i][j] = u32x4_v{0u, 0u, 0u, 0u};
                if (v < KEYS / 2 * VEC && kk <= kmax && e0 < p.vdim) vr[i][j] = *(const u32x4_v*)(vc + ((size_t)kk * vpitch + (size_t)g * p.vdim + e0) * 2);
            }
        }
    };
    const uint32_t kstep = SPLIT ? KEYS * gridDim.z : KEYS, kfirst = kmin + (SPLIT ? KEYS * blockIdx.z : 0);
    if (AHEAD && kfirst <= kmax) fetch(kfirst);
    for (uint32_t kb0 = kfirst; kb0 <= kmax; kb0 += kstep) {
        if (!AHEAD) fetch(kb0);
        __syncthreads(); // the stretch before has been read
#pragma unroll
        for (int i = 0; i < KN; ++i) {
            const uint32_t v = tid + i * T;
            if (v < KEYS * VEC) *(u32x4_v*)(s_k + v / VEC * KP + v % VEC * 16) = kr[i];
        }
#pragma unroll
        for (int i = 0; i < VN; ++i) { // two keys' elements side by side: 16 lanes write 64 bytes of a transposed row
            const uint32_t v = tid + i * T;
            if (v < KEYS / 2 * VEC) {
                uint8_t* to = s_vt + (v / (16 * VEC) * RP + v / 16 % VEC * 8) * TP + v % 16 * 4;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    *(uint32_t*)(to + (2 * e) * TP) = (vr[i][0][e] & 0xFFFFu) | (vr[i][1][e] << 16);
                    *(uint32_t*)(to + (2 * e + 1) * TP) = (vr[i][0][e] >> 16) | (vr[i][1][e] & 0xFFFF0000u);
                }
            }
        }
        if (AHEAD && kb0 + kstep <= kmax) fetch(kb0 + kstep);
        __syncthreads();
        const uint32_t kb = kb0 + 32 * kg;
        if (!wave_on || kb > wave_hi || kb + 31 < wave_lo) continue; // (wave-uniform; the barriers above are reached by every wave)
        f32x16_t st;
#pragma unroll
        for (int r = 0; r < 16; ++r) st[r] = 0.0f;
#pragma unroll
        for (int s = 0; s < 2 * NB; ++s) {
            const u32x4_t a = *(const u32x4_t*)(s_k + (32 * kg + l32) * KP + (s * 16 + half * 8) * 2);
            st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, qh[s]), st, 0, 0, 0);
            st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, ql[s]), st, 0, 0, 0);
        }
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t key = kb + (r & 3) + 8 * (r >> 2) + 4 * half;
            const bool ok = valid && key >= lo && key <= t;
            float sc = st[r] * hscale;
            if (p.soft_cap != 0.0f) { // cap * tanh(s / cap), tanh(x) = 1 - 2 / (1 + e^(2x))
                const float e2 = fast_exp(2.0f * sc * inv_cap);
                sc = p.soft_cap * (1.0f - 2.0f / (1.0f + e2));
            }
            if (p.dist_bias && ok) sc += p.dist_bias[(size_t)min(t - key, p.dist_rows - 1) * p.heads + head];
            st[r] = ok ? sc : -INFINITY;
            mx = fmaxf(mx, st[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m_run, mx);
        const float corr = fast_exp(m_run - m_new);
        float psum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            st[r] = fast_exp(st[r] - m_new); // masked: exp(-inf) = 0
            psum += st[r];
        }
        psum += __shfl_xor(psum, 32, 64);
        l_run = fmaf(l_run, corr, psum);
        m_run = m_new;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[b][r] *= corr;
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
            uint32_t hw[4], lwv[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) split_bf16(st[8 * s2 + 2 * e], st[8 * s2 + 2 * e + 1], hw[e], lwv[e]);
            const u32x4_t hi{hw[0], hw[1], hw[2], hw[3]}, lw{lwv[0], lwv[1], lwv[2], lwv[3]};
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const uint8_t* cr = s_vt + (kg * RP + b * 32 + l32) * TP + (16 * s2 + 4 * half) * 2;
                const u32x2_v c0 = *(const u32x2_v*)cr, c1 = *(const u32x2_v*)(cr + 16);
                const u32x4_t cf{c0.x, c0.y, c1.x, c1.y};
                o[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, cf), __builtin_bit_cast(bf16x8_t, hi), o[b], 0, 0, 0);
                o[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, cf), __builtin_bit_cast(bf16x8_t, lw), o[b], 0, 0, 0);
            }
        }
    }
    if (KG > 1) { // the groups' results: [group - 1][item block][value][lane], behind them the maxima and sums
        float* s_o = (float*)smem;
        constexpr int PER = (16 * NB + 2) * 64;
        __syncthreads();
        if (kg) {
            float* mine = s_o + ((kg - 1) * IW + wave) * PER + lane;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) mine[(b * 16 + r) * 64] = o[b][r];
            mine[16 * NB * 64] = m_run, mine[(16 * NB + 1) * 64] = l_run;
        }
        __syncthreads();
        if (kg) return;
#pragma unroll
        for (int other = 0; other < KG - 1; ++other) {
            const float* theirs = s_o + (other * IW + wave) * PER + lane;
            const float m_o = theirs[16 * NB * 64], l_o = theirs[(16 * NB + 1) * 64], m_new = fmaxf(m_run, m_o), a = fast_exp(m_run - m_new), c = fast_exp(m_o - m_new);
            l_run = l_run * a + l_o * c, m_run = m_new;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[b][r] = fmaf(theirs[(b * 16 + r) * 64], c, o[b][r] * a);
        }
    }
    if (!valid) return;
    if (SPLIT) {
        float* ws = p.split_ws + (((size_t)(sp.row0 + row) * p.heads + head) * gridDim.z + blockIdx.z) * (RP + 4);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4)
                *(f32x4_v*)(ws + b * 32 + 8 * g4 + 4 * half) = f32x4_v{o[b][4 * g4], o[b][4 * g4 + 1], o[b][4 * g4 + 2], o[b][4 * g4 + 3]};
        if (half == 0) ws[RP] = m_run, ws[RP + 1] = l_run;
        return;
    }
    float inv = p.out_scale / l_run;
    if (p.gate) inv *= 1.0f / (1.0f + expf(-p.gate[(size_t)(sp.row0 + row) * p.ldgate + head]));
    float* out = p.out + (size_t)(sp.row0 + row) * p.ldo + (size_t)head * p.vdim;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
            const uint32_t col = b * 32 + 8 * g4 + 4 * half;
            if (col < p.vdim) *(f32x4_v*)(out + col) = f32x4_v{o[b][4 * g4] * inv, o[b][4 * g4 + 1] * inv, o[b][4 * g4 + 2] * inv, o[b][4 * g4 + 3] * inv};
        }
}

// a workgroup per item: out = sum_s e^(m_s - M) O_s / sum_s e^(m_s - M) l_s over the splits, in split order (a split that saw no key has l = 0 and m = -1e30).  (The step form's merge, for up to 32
// shares and with a norm beside it, is slower behind this form: 64 heads on 8 of 64, 4 rows, window 1024 11.7 us in all for 10.7.)
// (gate: the item's result times sigmoid(gate[row, head]), item = row * heads + head)
__global__ void __launch_bounds__(128) window_attention_mfma_merge_kernel(const float* ws, float* out, uint32_t splits, uint32_t vdim, uint32_t rp, const float* gate, uint32_t ldgate,
                                                                     uint32_t heads, uint32_t ldo, float out_scale) {
    const uint32_t item = blockIdx.x, tid = threadIdx.x;
    const float* base = ws + (size_t)item * splits * (rp + 4);
    // the splits' weights once, a lane per split (at most 64 splits); the sums over the splits run in split order
    __shared__ float s_w[64], s_l[64];
    if (tid < 64) {
        const float m = tid < splits ? base[(size_t)tid * (rp + 4) + rp] : -1.0e30f;
        s_l[tid] = tid < splits ? base[(size_t)tid * (rp + 4) + rp + 1] : 0.0f;
        s_w[tid] = fast_exp(m - wave_max(m));
    }
    __syncthreads();
    float den = 0.0f;
    for (uint32_t s = 0; s < splits; ++s) den = fmaf(s_w[s], s_l[s], den);
    if (gate) den *= 1.0f + expf(-gate[(size_t)(item / heads) * ldgate + item % heads]);
    for (uint32_t c = tid; c < vdim; c += 128) {
        float acc = 0.0f;
#pragma unroll 8
        for (uint32_t s = 0; s < splits; ++s) acc = fmaf(s_w[s], base[(size_t)s * (rp + 4) + c], acc);
        out[(size_t)(item / heads) * ldo + (size_t)(item % heads) * vdim + c] = acc / den * out_scale;
    }
}

uint32_t blocks_of(const WindowAttentionParams& p) {
    const uint32_t w = p.dim > p.vdim ? p.dim : p.vdim;
    return w <= 32 ? 1 : w <= 64 ? 2 : w <= 128 ? 4 : 0;
}

} // namespace

size_t window_attention_split_ws_bytes(uint32_t rows, uint32_t heads, uint32_t splits) { return (size_t)rows * heads * splits * (128 + 4) * 4; }

// A workgroup that has one or two stretches of 32 keys to walk is through before one with a stretch of 128 has staged it and its four waves have met; with more of them the four
// waves are the faster walkers.  How few it can have is how many workgroups run at once: one a CU.  Heads of 128, 4 key / value heads, us a launch with its merge, stretches of 32 /
// of 128: one sequence, window 40 9.8 / 14.0, 128 10.5 / 14.4, 512 (16 splits) 10.1 / 15.4 (4), 1024 (16) 12.6 / 14.6 (8); 8 sequences, window 256 (8) 10.5 / 14.8 (2),
// 512 (8) 13.0 / 15.1 (4), 1024 (8) 18.3 / 14.1 (8); 32 sequences, window 128 (2) 13.3 / 14.5 (2), 256 (2) 18.5 / 14.6 (2).  Up to 32 keys the simple form is as fast.
static float split_us(const WindowAttentionParams& p, uint32_t seen) { // with the merge: a workgroup's stretches, the work over the chip's units of 256, the workgroups, and what the merge adds
    struct Cost {
        float launch, stretch, work, workgroups, shares;
    };
    const bool wide = blocks_of(p) > 2, short_stretches = p.split_items == 128;
    const Cost us = short_stretches ? (wide ? Cost{7.25f, 2.69f, -1.64f, 4.34f, 0.026f} : Cost{7.2f, 1.85f, -0.37f, 1.08f, 0.146f}) : (wide ? Cost{9.0f, 2.1f, 4.17f, 4.34f, 0.026f} : Cost{8.0f, 1.43f, 1.52f, 1.08f, 0.146f});
    const uint32_t stretches = short_stretches ? (seen + 31) / 32 : (seen + 127) / 128;
    const float units = (float)(p.rows * p.kv_heads) / 256.0f;
    return us.launch + us.stretch * (float)((stretches + p.splits - 1) / p.splits) + units * (us.work * (float)stretches + us.workgroups * (float)p.splits) + us.shares * 1e-3f * (float)p.rows * (float)(p.heads * p.splits);
}
// One row a sequence: the step form (k_window_attention_step.hip) or this one.  The step form reads a key once per four query heads of its key / value head, this one once, and its tiles are filled the better the
// more of those there are; its shares are cut for `keys`, however few a pass has.  Up to four of them, or over up to 224 keys, the step form is the faster one.  Else what either takes is estimated, from the
// keys that the pass' rows do see where it knows them (a captured one does not: up to 1000).  Us, this form and the step form: 24 heads on 2 of 128, 48 rows behind 150 / 700 / 2000 keys, no window 46 / 12,
// 52 / 40, 66 / 102; 64 on 8 of 64, window 1024, 6 rows 11.5 / 14.1, 32 rows 35.6 / 31.4.  8580 passes of five query heads and more: within 0.5 % of the faster form on the average, 141 off by more than
// 10 %, by at most 24 %.
void window_attention_split_keys(WindowAttentionParams& p, uint32_t keys, uint32_t num_cus) {
    WindowAttentionParams step = p;
    step.split_items = 0, step.splits = 1; // (one share: whether it takes the shape at all)
    const uint32_t blocks = (keys + 31) / 32, at_once = num_cus / std::max(1u, p.tiles * p.kv_heads), splits = std::min(blocks, std::max(2u, std::min(16u, at_once)));
    if (blocks <= 2 * splits) p.split_items = 128, p.splits = splits;
    else p.split_items = 32, p.splits = std::min(16u, std::max(2u, (keys + 127) / 128));
    if (!window_attention_step_supported(step)) return;
    step.splits = window_attention_step_splits(p, keys, num_cus);
    if (p.split_ws) step.splits = std::max<uint32_t>(1, std::min<size_t>(step.splits, p.split_ws_bytes / window_attention_split_ws_bytes(p.rows, p.heads, 1)));
    const uint32_t seen = std::min(keys, p.keys ? p.keys : 1000u);
    if (p.heads / p.kv_heads <= 4 || keys <= 224 || (p.split_ws && !window_attention_mfma_supported(p)) || window_attention_step_us(step, seen) <= split_us(p, seen)) p = step;
}

// bf16 caches, head widths that are multiples of 8 up to 128 (16-byte rows); prompt-sized passes, or a decode-sized pass with a workspace to split its keys
// (without one a decode step's few items would walk all their keys in one nearly empty workgroup: the simple form does that better)
static bool use_split(const WindowAttentionParams& p) {
    return p.splits > 1 && p.splits <= 64 && p.tiles32 && p.split_ws && p.split_ws_bytes >= window_attention_split_ws_bytes(p.rows, p.heads, p.splits);
}

bool window_attention_mfma_supported(const WindowAttentionParams& p) {
    const bool split = use_split(p);
    return p.cache_bf16 && blocks_of(p) && p.dim % 8 == 0 && p.vdim % 8 == 0 && p.ldq % 4 == 0 && p.ldo % 4 == 0 && p.kv_heads && p.heads % p.kv_heads == 0 && p.nseq && p.tiles &&
           (split || p.rows >= 16 * p.nseq) && p.kv_heads <= 65535 && ((uintptr_t)p.q & 15) == 0 && ((uintptr_t)p.out & 15) == 0;
}

template <int NB, int IW, int KG, bool SPLIT, bool AHEAD = true> static uzu_status launch(hipStream_t s, const WindowAttentionParams& p) {
    constexpr size_t stage = (size_t)32 * KG * (32 * NB * 2 + 16) + (size_t)KG * 32 * NB * 80, meet = (size_t)(KG - 1) * IW * (16 * NB + 2) * 256, lds = stage > meet ? stage : meet;
    static LdsLimit lim;
    UZU_REQUIRE(raise_lds_limit(lim, (const void*)window_attention_mfma_kernel<NB, IW, KG, SPLIT, AHEAD>, lds), "window_attention_mfma: %zu bytes of LDS are not available", lds);
    return launch_check([&] { hipLaunchKernelGGL((window_attention_mfma_kernel<NB, IW, KG, SPLIT, AHEAD>), dim3(IW == 1 ? p.tiles32 : p.tiles, p.kv_heads, SPLIT ? p.splits : 1), dim3(64 * IW * KG), lds, s, p); },
                        SPLIT ? "window_attention_mfma_split" : "window_attention_mfma");
}

uzu_status window_attention_mfma(hipStream_t s, const WindowAttentionParams& p) {
    UZU_REQUIRE(window_attention_mfma_supported(p), "window_attention: the matrix-core form does not take this shape");
    const uint32_t nb = blocks_of(p);
    if (use_split(p)) {
        if (p.split_items == 128) UZU_PROPAGATE(nb == 1 ? (launch<1, 4, 1, true>(s, p)) : nb == 2 ? (launch<2, 4, 1, true>(s, p)) : (launch<4, 4, 1, true>(s, p)));
        else UZU_PROPAGATE(nb == 1 ? (launch<1, 1, 4, true>(s, p)) : nb == 2 ? (launch<2, 1, 4, true>(s, p)) : (launch<4, 1, 4, true>(s, p)));
        return launch_check([&] { hipLaunchKernelGGL(window_attention_mfma_merge_kernel, dim3(p.rows * p.heads), dim3(128), 0, s, (const float*)p.split_ws, p.out, p.splits, p.vdim, 32 * nb, p.gate, p.ldgate, p.heads, p.ldo, p.out_scale); },
                            "window_attention_merge");
    }
    // Prompts with more tiles than CUs: a second tile on the CU covers a wave's waits as the second key group does, and the groups have to meet.  Us, one group and two: heads of 64, 2048
    // rows of 32 heads on 8 (512 tiles), window 64 / 256 / 512 / none 16.3 / 30.8 / 50.0 / 158 and 21.5 / 35.3 / 53.3 / 157; 1500 rows of 64 on 8 (752), 64 / 512 / none 21.8 / 61.1 / 124 and
    // 30.2 / 76.2 / 146; fewer tiles, 1500 rows of 32 on 8 (376), 64 / 128 / 256 14.5 / 19.7 / 29.4 and 19.9 / 24.6 / 33.8, longer keys no better than the two groups.  Heads of 128 do not
    // fit a second tile and its look-ahead (window 512, 512 tiles: 104 and 71.4): without the look-ahead, over short windows, 376 / 512 / 1024 tiles window 64 24.7 / 25.4 / 55.8 and 32.7 /
    // 33.2 / 72.5, window 256 42.5 / 44.8 / 84.9 and 46.2 / 50.0 / 103.
    const uint32_t seen = p.window && p.chunk ? std::min(p.window, p.chunk) : std::max(p.window, p.chunk);
    const uint64_t workgroups = (uint64_t)p.tiles * p.kv_heads;
    if (nb == 2 && (workgroups >= 512 || (workgroups > 256 && seen && seen <= 256))) return launch<2, 4, 1, false>(s, p);
    if (nb == 4 && workgroups > 256 && seen && seen <= 256) return launch<4, 4, 1, false, false>(s, p);
    return nb == 1 ? launch<1, 4, 2, false>(s, p) : nb == 2 ? launch<2, 4, 2, false>(s, p) : launch<4, 4, 2, false>(s, p);
}

} // namespace k
} // namespace uzu
