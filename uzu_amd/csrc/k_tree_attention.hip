// k_tree_attention.hip -- attention of a speculated tree's rows on the matrix cores, for gfx950.
//
// Semantics: AttentionSinglePass with is_trie (attention_single_pass.rs:37-127, mask.rs:21-29): a node sees every cached key and, among the tree's own, those whose
// {trie_start, trie_end} holds it.  A pass has 2 .. 32 nodes and a context of any length, and the keys are the same for all of them: what bounds it is the way from launch to
// first result, not the 1.5 MB of keys and values of 1500 positions (0.3 us at the copy rate).  So:
//   * a column of the products is a (head of the kv head's group, node) pair, 32 to a tile, and a workgroup has two tiles: 13 nodes of four heads are one workgroup a share
//     of the keys, which reads them once (a workgroup a node read them 13 times and spent a butterfly on every key);
//   * share z of up to 64 has the tiles z, z + shares, ... of 32 keys: the first tile's rows, the queries, the tree and the context's length are all requested at once, since
//     no address of them hangs on the length (the caches' memory bounds them);
//   * waves = (column tile, half of the head's elements): both halves work the scores out for themselves, which is cheaper than handing them over;
//   * the probabilities enter the second product as three bf16 terms, which hold all 24 bits of them, and the queries, keys and values are bf16: every product is exact
//     and the sums are in f32, as they are in the vector form (k_attention.hip);
//   * a key of another branch has weight zero, but zero times a value that is not finite is none: where that shows, the merge makes a share's sum again from the visible keys alone;
//   * partial results lie as [column tile][share][element][32 columns], so that both launches move whole lines.
// Layout of the operands as in k_attention_mfma.hip: scores transposed, so that a lane owns a column.
#include "device_utils.h"
#include "silu_near.h"
#include "tree_pass.h"

namespace uzu {
namespace k {

namespace {
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;

constexpr uint32_t kKeys = 32, kColumns = 32, kNodes = 32; // keys and columns of a tile (a workgroup: two tiles of columns)

__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    const bf16x2_t v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ f32x16_t mfma(const u32x4_v& a, const u32x4_v& b, const f32x16_t& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// grid (kv heads x pairs of column tiles, shares), 256 threads.  13 nodes of 8 heads of 256 behind 1500 keys: 7.9 us, of which the operands' trip is 2 and a tile's products 1.7; the
// vector form took 18.8 in front of its merge (4.7) and the gate (4.7).  64 shares against 32: half the tiles one behind the other, twice the partial results, 0.2 us less.
template <int HD>
__global__ void __launch_bounds__(256) tree_attention_kernel(AttentionParams a, uint32_t pairs, uint32_t key_rows, float* __restrict__ partials, float* __restrict__ sums,
                                                             float* __restrict__ maxs) {
    constexpr int KP = HD * 2 + 16, VP = kKeys * 2 + 8; // row pitches in bytes: conflict-free reads of 16 and of 8 bytes
    constexpr int NS = HD / 16, HB = HD / 64, VEC = HD / 8;
    constexpr int QN = 2 * kColumns * VEC / 256, KN = (kKeys * VEC + 255) / 256, VN = (kKeys / 2 * VEC + 255) / 256;
    __shared__ __attribute__((aligned(16))) uint8_t s_q[2 * kColumns * KP], s_k[2][kKeys * KP], s_v[2][HD * VP];
    const uint32_t tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5, wave = __builtin_amdgcn_readfirstlane(tid >> 6), tile = wave & 1, part = wave >> 1;
    const uint32_t n = a.suffix_length, columns = a.gqa_factor * n, kv_head = blockIdx.x / pairs, pair = blockIdx.x - kv_head * pairs, share = blockIdx.y, shares = gridDim.y;
    const uint32_t first = (2 * pair + tile) * kColumns; // this wave's first column; column c = (head c / n of the group, node c % n)

    // staging role: 16 bytes of a key; 16 bytes of two neighbouring keys' values
    const uint16_t* keys = (const uint16_t*)a.keys + (size_t)kv_head * a.k_head_stride;
    const uint16_t* values = (const uint16_t*)a.values + (size_t)kv_head * a.v_head_stride;
    u32x4_v kst[KN], vst[VN][2];
    auto load = [&](uint32_t t) {
#pragma unroll
        for (int r = 0; r < KN; ++r) {
            const uint32_t v = min(tid + r * 256, (uint32_t)(kKeys * VEC - 1)), i = min(t * kKeys + v / VEC, key_rows - 1);
            kst[r] = *(const u32x4_v*)(keys + (size_t)i * a.k_seq_stride + v % VEC * 8);
        }
#pragma unroll
        for (int r = 0; r < VN; ++r)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t v = min(tid + r * 256, (uint32_t)(kKeys / 2 * VEC - 1)), i = min(t * kKeys + v % 16 * 2 + j, key_rows - 1);
                vst[r][j] = *(const u32x4_v*)(values + (size_t)i * a.v_seq_stride + v / 16 * 8);
            }
    };
    auto store = [&](uint32_t t, uint32_t length, int buf) { // (rows past the last key may hold anything: a probability of 0 does not help against a NaN)
        const u32x4_v zero = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int r = 0; r < KN; ++r) {
            const uint32_t v = tid + r * 256;
            if (kKeys * VEC % 256 && v >= (uint32_t)(kKeys * VEC)) continue;
            *(u32x4_v*)(s_k[buf] + v / VEC * KP + v % VEC * 16) = t * kKeys + v / VEC < length ? kst[r] : zero;
        }
#pragma unroll
        for (int r = 0; r < VN; ++r) {
            const uint32_t v = tid + r * 256, i = t * kKeys + v % 16 * 2;
            if (kKeys / 2 * VEC % 256 && v >= (uint32_t)(kKeys / 2 * VEC)) continue;
            const u32x4_v v0 = i < length ? vst[r][0] : zero, v1 = i + 1 < length ? vst[r][1] : zero;
            uint8_t* to = s_v[buf] + v / 16 * 8 * VP + v % 16 * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                *(uint32_t*)(to + (2 * e) * VP) = (v0[e] & 0xFFFFu) | (v1[e] << 16);
                *(uint32_t*)(to + (2 * e + 1) * VP) = (v0[e] >> 16) | (v1[e] & 0xFFFF0000u);
            }
        }
    };
    uint2 range = make_uint2(1u, 0u); // node l32's range (no node is in this one), in every wave; requested first, since the loads come back in their order
    if (l32 < n) range = make_uint2(a.trie[3 * l32], a.trie[3 * l32 + 1]);
    load(share);
    u32x4_v qst[QN]; // the columns of a kv head are consecutive rows of the queries
    {
        const uint16_t* q = (const uint16_t*)a.queries + (size_t)kv_head * columns * HD;
#pragma unroll
        for (int r = 0; r < QN; ++r) {
            const uint32_t v = tid + r * 256;
            qst[r] = *(const u32x4_v*)(q + (size_t)min(2 * pair * kColumns + v / VEC, columns - 1) * HD + v % VEC * 8);
        }
    }
    const uint32_t length = a.sequence_length + (a.dyn ? *a.dyn : 0u), prefix = length - n, tiles = (length + kKeys - 1) / kKeys;
    const size_t at = ((size_t)kv_head * 2 * pairs + 2 * pair + tile) * shares + share; // this wave's partial result
    if (share >= tiles) { // no key of this share: the merge reads its maximum alone
        if (part == 0 && half == 0) sums[at * kColumns + l32] = 0.f, maxs[at * kColumns + l32] = -INFINITY;
        return;
    }
    // bit j: this lane's node sees the tree's key j.  A node's bits are one comparison of all lanes, made while the rows are on their way (a lane that read the ranges of 32 keys
    // out of LDS behind the scores took 7500 cycles of the last share's 19600)
    const uint32_t node = (first + l32) % n;
    uint32_t seen = 0;
    for (uint32_t q0 = 0; q0 < n; q0 += 8)
#pragma unroll
        for (uint32_t q = q0; q < q0 + 8; ++q) {
            const uint32_t keys_of_q = (uint32_t)__builtin_amdgcn_ballot_w64(q >= range.x && q <= range.y);
            seen = node == q ? keys_of_q : seen;
        }
#pragma unroll
    for (int r = 0; r < QN; ++r) {
        const uint32_t v = tid + r * 256;
        *(u32x4_v*)(s_q + v / VEC * KP + v % VEC * 16) = qst[r];
    }
    store(share, length, 0);
    __syncthreads();
    u32x4_v qf[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) qf[s] = *(const u32x4_v*)(s_q + (tile * kColumns + l32) * KP + half * 16 + s * 32);
    f32x16_t o[HB];
#pragma unroll
    for (int b = 0; b < HB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[b][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f; // l_run: this lane's half of the keys
    int buf = 0;
    for (uint32_t t = share; t < tiles; t += shares, buf ^= 1) {
        const bool more = t + shares < tiles;
        if (more) load(t + shares);
        if (first < columns) {
            // every operand of the tile is on its way before the first product (left to the order below, reads were waited for two by two: 4400 cycles a tile, now 3800)
            u32x4_v kf[NS], vf[2][HB];
            const uint8_t* k = s_k[buf] + l32 * KP + half * 16;
#pragma unroll
            for (int s = 0; s < NS; ++s) kf[s] = *(const u32x4_v*)(k + s * 32);
#pragma unroll
            for (int step = 0; step < 2; ++step)
#pragma unroll
                for (int b = 0; b < HB; ++b) { // a lane's element of the head: keys 16 step + 4 half + {0..3} and 8 further
                    const uint8_t* v = s_v[buf] + ((part * HB + b) * 32 + l32) * VP + (16 * step + 4 * half) * 2;
                    const u32x2_v lo = *(const u32x2_v*)v, hi = *(const u32x2_v*)(v + 16);
                    vf[step][b] = u32x4_v{lo.x, lo.y, hi.x, hi.y};
                }
            __builtin_amdgcn_sched_barrier(0);
            f32x16_t acc;
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
            for (int s = 0; s < NS; ++s) acc = mfma(kf[s], qf[s], acc);
            float score[16], m_mine = -INFINITY; // (this lane's keys: (r & 3) + 8 (r >> 2) + 4 half)
            if (t * kKeys + kKeys <= prefix) {
#pragma unroll
                for (int r = 0; r < 16; ++r) score[r] = a.scale * acc[r];
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t key = t * kKeys + 4 * half + (r & 3) + 8 * (r >> 2), j = key - prefix;
                    score[r] = key < prefix || (key < length && (seen >> (j & 31) & 1)) ? a.scale * acc[r] : -INFINITY;
                }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) m_mine = fmaxf(m_mine, score[r]);
            const float m_new = fmaxf(m_run, fmaxf(m_mine, __shfl_xor(m_mine, 32, 64)));
            const float alpha = m_new == -INFINITY ? 1.0f : fast_exp(m_run - m_new), m_ref = m_new == -INFINITY ? 0.f : m_new; // (-inf: no key seen, or NaNs)
            float sum = 0.f;
            u32x4_v p[3][2]; // the probabilities' three terms of two k16 steps
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const float p0 = fast_exp(score[r] - m_ref), p1 = fast_exp(score[r + 1] - m_ref);
                sum += p0 + p1;
                const float h0 = round_bf16(p0), h1 = round_bf16(p1), r0 = p0 - h0, r1 = p1 - h1, i0 = round_bf16(r0), i1 = round_bf16(r1);
                p[0][r / 8][r / 2 % 4] = pack2(h0, h1), p[1][r / 8][r / 2 % 4] = pack2(i0, i1), p[2][r / 8][r / 2 % 4] = pack2(r0 - i0, r1 - i1);
            }
            l_run = l_run * alpha + sum, m_run = m_new;
            if (t != share) {
#pragma unroll
                for (int b = 0; b < HB; ++b)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[b][r] *= alpha;
            }
#pragma unroll
            for (int step = 0; step < 2; ++step)
#pragma unroll
                for (int term = 0; term < 3; ++term)
#pragma unroll
                    for (int b = 0; b < HB; ++b) o[b] = mfma(vf[step][b], p[term][step], o[b]);
        }
        if (more) store(t + shares, length, buf ^ 1);
        lds_barrier();
    }
    const float l = l_run + __shfl_xor(l_run, 32, 64);
    if (first >= columns) return; // (columns past the last are nobody's; a tile past the last has no place among the partial results either)
    float* to = partials + (at * HD + part * (HD / 2)) * kColumns + l32;
#pragma unroll
    for (int b = 0; b < HB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) to[(b * 32 + (r & 3) + 8 * (r >> 2) + 4 * half) * kColumns] = o[b][r];
    if (part == 0 && half == 0) sums[at * kColumns + l32] = l, maxs[at * kColumns + l32] = m_run;
}

// A share's sum for one element of a column, from the keys that its node sees, one after the other
template <int HD>
__device__ __forceinline__ float visible_sum(const AttentionParams& a, uint32_t kv_head, uint32_t column, uint32_t node, uint32_t element, uint32_t share, uint32_t shares, float top) {
    const uint32_t n = a.suffix_length, length = a.sequence_length + (a.dyn ? *a.dyn : 0u), prefix = length - n;
    const uint16_t* q = (const uint16_t*)a.queries + ((size_t)kv_head * a.gqa_factor * n + column) * HD;
    const uint16_t *keys = (const uint16_t*)a.keys + (size_t)kv_head * a.k_head_stride, *values = (const uint16_t*)a.values + (size_t)kv_head * a.v_head_stride + element;
    float sum = 0.f;
    for (uint32_t t = share; t * kKeys < length; t += shares)
        for (uint32_t i = t * kKeys; i < min(t * kKeys + kKeys, length); ++i) {
            if (i >= prefix && !(node >= a.trie[3 * (i - prefix)] && node <= a.trie[3 * (i - prefix) + 1])) continue;
            float score = 0.f;
            for (uint32_t d = 0; d < HD; ++d) score = fmaf(bf16_to_f32(q[d]), bf16_to_f32(keys[(size_t)i * a.k_seq_stride + d]), score);
            sum = fmaf(fast_exp(a.scale * score - top), bf16_to_f32(values[(size_t)i * a.v_seq_stride]), sum);
        }
    return sum;
}

// The rows from their shares, and the gate: a workgroup has 8 elements of a column tile, a thread one of a column, everything requested before any of it is used.  6.7 us
// behind 1500 keys (48 shares of 128 KB), where the two-pass form's second kernel and the gate's were 9.4.
// grid (kv heads x column tiles, head_dim / 8), 256 threads
template <int HD>
__global__ void __launch_bounds__(256) tree_attention_merge_kernel(AttentionParams a, const float* __restrict__ partials, const float* __restrict__ sums, const float* __restrict__ maxs,
                                                                   uint16_t* __restrict__ out, const uint16_t* __restrict__ gate, uint32_t tiles, uint32_t pairs, uint32_t shares) {
    constexpr uint32_t head_dim = HD;
    const uint32_t n = a.suffix_length, group_heads = a.gqa_factor, heads = a.num_heads, sequence_length = a.sequence_length;
    const uint32_t* const dyn = a.dyn;
    const uint32_t used = min(shares, (sequence_length + (dyn ? *dyn : 0u) + kKeys - 1) / kKeys); // shares with keys: nothing of the others but their maxima has been written
    constexpr uint32_t P = kTreeAttentionShares / 8;
    __shared__ float s_max[8][kColumns], s_sum[8][kColumns], s_w[kTreeAttentionShares][kColumns];
    __shared__ uint64_t s_exp_tab[32];
    const uint32_t tid = threadIdx.x, c = tid % kColumns, e = tid / kColumns, kv_head = blockIdx.x / tiles, tile = blockIdx.x - kv_head * tiles, element = blockIdx.y * 8 + e;
    const uint32_t column = tile * kColumns + c, columns = group_heads * n, head = kv_head * group_heads + min(column, columns - 1) / n, node = min(column, columns - 1) % n;
    const size_t at = ((size_t)kv_head * 2 * pairs + tile) * shares, row = (size_t)node * heads + head;
    float m[P], l[P], v[kTreeAttentionShares];
#pragma unroll
    for (uint32_t i = 0; i < P; ++i) { // (shares come in eights, each with its maximum and sum)
        const size_t share = at + e + 8 * i;
        m[i] = -INFINITY, l[i] = 0.f;
        if (8 * i < used) m[i] = maxs[share * kColumns + c], l[i] = sums[share * kColumns + c];
    }
    const uint16_t g = gate ? gate[row * head_dim + element] : (uint16_t)0;
#pragma unroll
    for (uint32_t i = 0; i < P; ++i)
        if (8 * i < used) {
#pragma unroll
            for (uint32_t b = 8 * i; b < 8 * i + 8; ++b) v[b] = partials[((at + b) * head_dim + element) * kColumns + c];
        }
    if (tid < 32) s_exp_tab[tid] = kExp2fTab[tid];
    __builtin_amdgcn_sched_barrier(0);
    float m_all = -INFINITY;
#pragma unroll
    for (uint32_t i = 0; i < P; ++i) m_all = fmaxf(m_all, m[i]);
    s_max[e][c] = m_all;
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) m_all = fmaxf(m_all, s_max[i][c]); // (a maximum does not depend on its order)
    float sum = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < P; ++i) {
        const float w = expf_glibc_tab(m[i] - m_all, s_exp_tab);
        s_w[e + 8 * i][c] = m[i] == -INFINITY ? -1.f : w, sum += l[i] * w; // (-1: no key seen, no elements written)
    }
    s_sum[e][c] = sum;
    __syncthreads();
    if (column >= columns) return;
    float l_all = 0.f, o = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) l_all += s_sum[i][c];
#pragma unroll
    for (uint32_t i = 0; i < P; ++i)
        if (8 * i < used) {
#pragma unroll
            for (uint32_t b = 8 * i; b < 8 * i + 8; ++b) {
                const float w = s_w[b][c];
                o += w < 0.f ? 0.f : v[b] * w;
            }
        }
    if (__builtin_expect(o != o && l_all == l_all, 0)) {
        o = 0.f;
        for (uint32_t b = 0; b < used; ++b) {
            const float w = s_w[b][c];
            if (w < 0.f) continue;
            float part = partials[((at + b) * head_dim + element) * kColumns + c];
            if (part != part) part = visible_sum<HD>(a, kv_head, column, node, element, b, shares, maxs[(at + b) * kColumns + c]);
            o += part * w;
        }
    }
    uint16_t bits = f32_to_bf16(o / l_all);
    if (gate) bits = scaled_sigmoid_bf16(bf16_to_f32(bits), bf16_to_f32(g), s_exp_tab);
    out[row * head_dim + element] = bits;
}
// kv heads x pairs of column tiles; the shares that put a workgroup on most of the compute units
uint32_t tree_pairs(uint32_t group_heads, uint32_t nodes) { return (group_heads * nodes + 2 * kColumns - 1) / (2 * kColumns); }
uint32_t tree_shares(uint32_t kv_heads, uint32_t pairs) {
    uint32_t shares = kTreeAttentionShares;
    while (shares > 8 && kv_heads * pairs * shares > kChipCus) shares >>= 1;
    return shares;
}
} // namespace

bool attention_tree_supported(const AttentionParams& a) {
    if (exact_mode() || !a.trie || a.dt != UZU_BF16 || !a.is_causal) return false;
    if (a.sinks || a.is_sliding_window || a.is_kv_cache_ring) return false; // (their masks stay with the vector form)
    if (!a.suffix_length || a.suffix_length > kNodes || !(a.head_dim == 64 || a.head_dim == 128 || a.head_dim == 256)) return false;
    if (!a.gqa_factor || a.num_heads % a.gqa_factor) return false;
    if (a.k_head_stride % 8 || a.k_seq_stride % 8 || a.v_head_stride % 8 || a.v_seq_stride % 8) return false;
    return (((uintptr_t)a.queries | (uintptr_t)a.keys | (uintptr_t)a.values) & 15) == 0; // rows are read 16 bytes at a time
}

// The vector form (k_attention.hip) has a workgroup per node and group of `gs` heads, and shares of the keys in its two passes alone.  Single pass: 3.4 us for heads by themselves, 4.3 in pairs, 6 in
// fours, and then 0.011 / 0.021 / 0.045 us a key of 64 / 128 / 256, half as much again in pairs; the tree form 7.8 / 8.4 / 9.5 us and next to nothing a key (heads by themselves, 13 nodes, us,
// single pass and tree: 16 of 128 behind 80 keys 5.4 / 8.5, 250 9.1 / 9.1, 600 20.9 / 10.4; 8 of 64 behind 250 6.4 / 8.3, 450 8.6 / 8.3): where the two meet is below, and groups of eight are slower from
// the first key on.  Two passes: what counts is how much work there is.  The tree form wants its columns filled, or the vector form's workgroups to be more than the chip holds.  Us, two passes
// and tree, 1500 and 4000 keys: 16 heads of 128, 4 nodes 9.9 / 11.8 and 15.4 / 19.4, 8 nodes 14.6 / 11.8 and 24.1 / 19.2; 32 on 8 of 128, 1 node 9.4 / 11.5 and 12.3 / 14.1, 3 nodes 12.6 / 10.8 and
// 18.4 / 13.4; 8 on 4 of 256, 6 nodes 11.5 / 12.4 and 19.0 / 16.0, 8 nodes 12.9 / 12.4 and 21.6 / 15.9; 8 on 2 of 256, 3 nodes 11.0 / 11.8 and 17.5 / 14.8, 4 nodes 11.1 / 11.8 and 17.6 / 14.7, with the gate
// 3 .. 4 us less for the tree form.
bool attention_tree_faster(uint32_t num_heads, uint32_t gqa_factor, uint32_t head_dim, uint32_t nodes, uint32_t keys, bool two_pass, bool gated) {
    uint32_t gs = 0; // heads of a workgroup of the vector form: 1 << gs
    while (gs < (head_dim >= 256 ? 2u : 3u) && gqa_factor % (2u << gs) == 0) ++gs;
    if (gs == 3) return true;
    if (!two_pass) {
        static constexpr uint32_t meet[3][3] = {{440, 240, 90}, {260, 160, 110}, {135, 90, 70}}; // [heads of 64, 128, 256][gs]
        return keys > meet[head_dim <= 64 ? 0 : head_dim <= 128 ? 1 : 2][gs];
    }
    const uint32_t rows = nodes * num_heads, columns = nodes * gqa_factor, half = gated ? 2 : 1;
    return rows >= 128 / half || (columns >= (head_dim >= 256 ? 16 : 12) / half && rows * head_dim > 6144 / half);
}

size_t attention_tree_columns(uint32_t num_heads, uint32_t gqa_factor, uint32_t nodes) {
    const uint32_t kv_heads = num_heads / gqa_factor, pairs = tree_pairs(gqa_factor, nodes);
    return (size_t)kv_heads * pairs * 2 * kColumns * tree_shares(kv_heads, pairs);
}

uzu_status attention_tree(hipStream_t s, const AttentionParams& a, uint32_t key_rows, float* partials, float* sums, float* maxs, void* out, const void* gate) {
    const uint32_t kv_heads = a.num_heads / a.gqa_factor, pairs = tree_pairs(a.gqa_factor, a.suffix_length), shares = tree_shares(kv_heads, pairs);
    const uint32_t tiles = (a.gqa_factor * a.suffix_length + kColumns - 1) / kColumns;
    const dim3 grid(kv_heads * pairs, shares);
    UZU_PROPAGATE(launch_check([&] {
        if (a.head_dim == 64) hipLaunchKernelGGL((tree_attention_kernel<64>), grid, dim3(256), 0, s, a, pairs, key_rows, partials, sums, maxs);
        else if (a.head_dim == 128) hipLaunchKernelGGL((tree_attention_kernel<128>), grid, dim3(256), 0, s, a, pairs, key_rows, partials, sums, maxs);
        else hipLaunchKernelGGL((tree_attention_kernel<256>), grid, dim3(256), 0, s, a, pairs, key_rows, partials, sums, maxs);
    }, "tree_attention"));
    return launch_check([&] {
#define UZU_TM(HD) hipLaunchKernelGGL(tree_attention_merge_kernel<HD>, dim3(kv_heads * tiles, HD / 8), dim3(256), 0, s, a, partials, sums, maxs, (uint16_t*)out, (const uint16_t*)gate, tiles, pairs, shares)
        if (a.head_dim == 64) UZU_TM(64);
        else if (a.head_dim == 128) UZU_TM(128);
        else UZU_TM(256);
#undef UZU_TM
    }, "tree_attention_merge");
}

} // namespace k
} // namespace uzu
