// k_attention_mfma.hip -- prefill attention on the bf16 matrix cores (flash-attention form) for gfx950.
//
// Reference semantics: AttentionSinglePass / TwoPass (BU/cpu/kernel/attention/attention_single_pass.rs:37-127,
// mask.rs:3-61): per (head, query) softmax(scale * q.k) over the visible keys (all cached keys + the causal part of
// the suffix), output [M, heads, hd] bf16.  The stand-alone VALU kernels (k_attention.hip) spend ~45 instructions per
// (query, key, head); at a 1024-token chunk that is the third-largest item of the prefill.  Here:
//
//   * a workgroup = one kv head x four wave tasks; a task is (32-query tile, q head of the kv head's GQA group), tasks are
//     numbered tile-major, so the four waves of a workgroup are four heads of one tile (GQA factor 4, 8, ...), two heads of two
//     tiles (factor 2), four tiles (factor 1) or whatever four consecutive tasks are (factor 3, 5, 6, 7: Qwen3-14B has 40 q /
//     8 kv heads) -- they share every K / V tile, staged once in LDS, and a wave skips the tiles past its own causal range;
//   * everything is computed TRANSPOSED so that a lane owns one query: S^T = K Q^T (A = K rows from LDS, B = Q^T from
//     registers), the C layout of v_mfma_f32_32x32x16_bf16 then gives a lane 16 key scores of ITS query (col = lane &
//     31), so the online-softmax statistics are per-lane scalars (one exchange with lane ^ 32 per tile for the
//     running maximum);  O^T = V^T P^T: the P^T operand is exactly those 16 registers (converted to bf16) -- no
//     shuffle, no LDS round trip -- and the O^T accumulator columns are again "this lane's query", so the rescale by
//     exp(m_old - m_new) and the final 1 / l are per-lane multiplies;
//   * V is stored transposed in LDS ([hd][key]): the contraction runs over keys, so a lane needs 8 keys of one hd
//     column; K stays [key][hd];
//   * q, k, v are bf16 already => every q.k product is exact in f32.  The probabilities are NOT bf16: they are fed
//     as hi + lo (two bf16 MFMAs, 16 significant bits), so the only arithmetic difference to the f32 reference is
//     the summation order.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "device_utils.h"
#include "attention_prefill.h"
#include "kernels.h"
#include "silu_near.h"

namespace uzu {
namespace k {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

namespace {
constexpr int TK = 32; // keys per tile (one MFMA block)
constexpr int TQ = 32; // queries per wave
constexpr uint32_t kMaxKeySplits = 12;

// How a launch's workgroups divide the keys.  A group of tasks (four consecutive ones) sees the keys in front of its last query, so equal numbers of shares would leave the last
// group's the longest by far: group y has a share per `quantum` stretches of keys that it was thought to see, and works out its shares from the keys that it does see.
struct KeyShares {
    uint32_t quantum; // stretches a share; 0: no shares, every group to its end by itself
    uint32_t prefix;  // cached keys, as far as the host knows
};
__host__ __device__ inline uint32_t key_stretches(const KeyShares& k, uint32_t y, uint32_t tpw, uint32_t gqa, uint32_t M, uint32_t stretch) {
    const uint32_t n_tasks = gqa * ((M + TQ - 1) / TQ), task = y * tpw + tpw - 1, end = ((task < n_tasks ? task : n_tasks - 1) / gqa + 1) * TQ;
    return (k.prefix + (end < M ? end : M) + stretch - 1) / stretch;
}
__host__ __device__ inline uint32_t key_shares(const KeyShares& k, uint32_t y, uint32_t tpw, uint32_t gqa, uint32_t M, uint32_t stretch) {
    if (!k.quantum) return 1;
    const uint32_t shares = (key_stretches(k, y, tpw, gqa, M, stretch) + k.quantum - 1) / k.quantum;
    return shares < kMaxKeySplits ? shares : kMaxKeySplits;
}

__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    const bf16x2_t v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
}
// value of lane ^ 32 (the other half of the wave): the one cross-half exchange per tile
__device__ __forceinline__ float other_half(float v) { return __shfl_xor(v, 32, 64); }
} // namespace

// grid: (kv heads, ceil(gqa * query tiles / tpw)); 256 KG threads.  Workgroups with the longest key ranges are numbered first.
// tpw = wave tasks per workgroup (4, 2 or 1): models with few heads (Qwen3.5-0.8B: 8 q heads -> 256 tasks per 1024-token chunk)
// would fill 64 CUs at four tasks per workgroup; with fewer tasks the idle waves still help staging the K / V tiles.
// Key split (few-head models: Qwen3.5-0.8B has 2 kv heads -> 64 workgroups of four tasks per 1024-token chunk): several workgroups share a
// task group (KeyShares), each takes an equal share of the key tiles ITS queries can see and leaves the unnormalised O^T, the running maximum and the
// sum as f32 partials ([split][query][head]); attention_prefill_merge_kernel folds them (the AttentionTwoPass2 step of the decode path).
// GEN: the general mask of mask.rs:3-61 without the trie -- sliding window, ring KV prefix (AttentionStateType::Ring: the prefix rows are a
// ring of `prefix` slots, key position = (prefix + i - ring_offset) mod prefix, live iff < ring_length) and attention sinks (the running
// maximum starts at the head's sink logit with a unit of mass: attention_single_pass.rs:70-74) -- evaluated per key on its POSITION; the
// plain causal instantiation keeps its one comparison per key.
// KG groups of four waves share a stretch of 32 KG keys, a wave takes its group's 32 of them, and the groups' unnormalised results meet in LDS at the end, in group order: the
// grid is about a workgroup per CU, and a wave alone on its SIMD waits for itself at every exponential (1021 rows of 32 heads of 128: 72 us with one group, 39 with
// two).  Heads of 256 need the registers of a wave alone.
// SEQS: several sequences, each with its own rows and cache, gridDim.x = kv heads x sequences and no key splits: the workgroups with the longest key ranges of all of them come first, and the
// short ones fill what a sequence by itself leaves idle (four of 1021 rows, 32 heads of 128: 4 x 39 us -> 99).
template <int HD, bool GEN, bool SEQS = false, int KG = HD <= 128 ? 2 : 1>
__global__ void __launch_bounds__(256 * KG) attention_prefill_mfma_kernel(AttentionParams a, uint16_t* out, uint32_t tpw, float* part_o, float* part_ml, std::conditional_t<SEQS, AttentionSeqs, KeyShares> more) {
    constexpr int KP = HD * 2 + 16;  // K tile row pitch in bytes (conflict-free ds_read_b128)
    constexpr int VP = TK * 2 + 8;   // V^T tile row pitch in bytes: 32 keys + 8 bytes of pad (conflict-free ds_read_b64)
    constexpr int NS = HD / 16;      // k16 steps of the QK^T contraction
    constexpr int NB = HD / 32;      // 32-row blocks of O^T
    constexpr int T = 256 * KG, KEYS = TK * KG, VEC = HD / 8;
    constexpr int KB = KEYS * KP, VB = KG * HD * VP; // a stretch's keys / values in LDS
    constexpr int PER = (16 * NB + 2) * 64;          // floats of a wave's result
    static_assert(KG == 1 || 4 * (KG - 1) * PER * 4 <= 2 * (KB + VB), "the groups' results fit where the keys and values were");
    __shared__ __attribute__((aligned(16))) uint8_t s_mem[2 * (KB + VB)];
    auto s_k = [&](int buf) { return s_mem + buf * KB; };
    auto s_vt = [&](int buf) { return s_mem + 2 * KB + buf * VB; };

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3, kg = __builtin_amdgcn_readfirstlane(tid >> 8), half = lane >> 5, l32 = lane & 31;
    const uint32_t M = a.suffix_length;
    uint32_t kv_head = blockIdx.x;
    if constexpr (SEQS) {
        const uint32_t kv_heads = a.num_heads / a.gqa_factor, seq = kv_head / kv_heads;
        kv_head -= seq * kv_heads;
        a.queries = more.queries[seq], a.keys = more.keys[seq], a.values = more.values[seq], a.dyn = more.dyn[seq], out = (uint16_t*)more.out[seq];
    }
    const uint32_t n_tasks = a.gqa_factor * ((M + TQ - 1) / TQ);
    uint32_t y = gridDim.y - 1 - blockIdx.y, share = 0, shares = 1; // heaviest (last query tiles) first
    if constexpr (!SEQS)
        if (more.quantum) {
            y = (n_tasks + tpw - 1) / tpw - 1, share = blockIdx.y;
            while (share >= (shares = key_shares(more, y, tpw, a.gqa_factor, M, KEYS))) share -= shares, --y;
        }
    const uint32_t task0 = y * tpw;
    const uint32_t task = task0 + wave;
    const bool wave_live = (uint32_t)wave < tpw && task < n_tasks;
    const uint32_t task_c = wave_live ? task : n_tasks - 1;
    const uint32_t head = kv_head * a.gqa_factor + task_c % a.gqa_factor;
    if constexpr (GEN) attention_resolve_dyn(a); // ring parameters / sequence length from the device-resident accepted-token count
    const uint32_t sequence_length = a.sequence_length + (a.dyn ? *a.dyn : 0u);
    const uint32_t prefix = sequence_length - M;
    const uint32_t suffix_position = (GEN && a.is_kv_cache_ring) ? a.ring_length : prefix; // attention_single_pass.rs:52-61
    const uint32_t q0 = (task_c / a.gqa_factor) * TQ; // first query of this wave
    const uint32_t qi = q0 + l32;                           // this lane's query (suffix index)
    const bool q_live = wave_live && qi < M;

    // ---- Q^T operand: lane = (query l32, hd half): 8 consecutive hd elements per k16 step, kept in registers
    u32x4_t qf[NS];
    {
        const uint16_t* qrow = (const uint16_t*)a.queries + ((size_t)head * M + (q_live ? qi : 0)) * HD + 8 * half;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const uint4 t = q_live ? *(const uint4*)(qrow + 16 * s) : make_uint4(0, 0, 0, 0);
            qf[s] = u32x4_t{t.x, t.y, t.z, t.w};
        }
    }

    // ---- staging role: thread -> 16 bytes of a key's row; 16 bytes of two neighbouring keys' values
    const uint16_t* kbase = (const uint16_t*)a.keys + (size_t)kv_head * a.k_head_stride;
    const uint16_t* vbase = (const uint16_t*)a.values + (size_t)kv_head * a.v_head_stride;
    constexpr int KN = KEYS * VEC / T, VN = (KEYS / 2 * VEC + T - 1) / T;
    u32x4_v kst[KN], vst[VN][2]; // native vectors + unconditional loads: stay in registers and in flight across lds_barrier()
    // keys visible to ANY query of the workgroup: 0 .. prefix + last query of its last live task (tasks are tile-major)
    const uint32_t last_tile = ((task0 + tpw - 1 < n_tasks ? task0 + tpw - 1 : n_tasks - 1) / a.gqa_factor + 1) * TQ;
    const uint32_t wg_last_q = (last_tile < M ? last_tile : M) - 1;
    const uint32_t key_end = prefix + wg_last_q + 1;
    const uint32_t n_tiles_all = (key_end + KEYS - 1) / KEYS; // (tiles of the workgroup: stretches of KEYS)
    const uint32_t per_share = (n_tiles_all + shares - 1) / shares;
    const uint32_t t_lo = min(share * per_share, n_tiles_all), n_tiles = min(t_lo + per_share, n_tiles_all); // this workgroup: tiles [t_lo, n_tiles)
    auto load_tile = [&](uint32_t t) {
        const u32x4_v zero = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int r = 0; r < KN; ++r) {
            const uint32_t v = tid + r * T, i = t * KEYS + v / VEC;
            const u32x4_v kk = *(const u32x4_v*)(kbase + (size_t)(i < key_end ? i : key_end - 1) * a.k_seq_stride + v % VEC * 8); // clamped row: masked keys get probability 0 anyway, zeroed for hygiene
            kst[r] = i < key_end ? kk : zero;
        }
#pragma unroll
        for (int r = 0; r < VN; ++r)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t v = min((uint32_t)(tid + r * T), (uint32_t)(KEYS / 2 * VEC - 1)), i = t * KEYS + v / (16 * VEC) * TK + v % 16 * 2 + j;
                const u32x4_v vv = *(const u32x4_v*)(vbase + (size_t)(i < key_end ? i : key_end - 1) * a.v_seq_stride + v / 16 % VEC * 8);
                vst[r][j] = i < key_end ? vv : zero;
            }
    };
    auto store_tile = [&](int buf) {
#pragma unroll
        for (int r = 0; r < KN; ++r) {
            const uint32_t v = tid + r * T;
            *(u32x4_v*)(s_k(buf) + v / VEC * KP + v % VEC * 16) = kst[r];
        }
        // V transposed, two keys' elements side by side: 16 lanes write 64 bytes of a row (element by element was 64 two-byte stores a thread, eight to a bank)
#pragma unroll
        for (int r = 0; r < VN; ++r) {
            const uint32_t v = tid + r * T;
            if (v >= (uint32_t)(KEYS / 2 * VEC)) continue;
            uint8_t* to = s_vt(buf) + (v / (16 * VEC) * HD + v / 16 % VEC * 8) * VP + v % 16 * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                *(uint32_t*)(to + (2 * e) * VP) = (vst[r][0][e] & 0xFFFFu) | (vst[r][1][e] << 16);
                *(uint32_t*)(to + (2 * e + 1) * VP) = (vst[r][0][e] >> 16) | (vst[r][1][e] & 0xFFFF0000u);
            }
        }
    };

    f32x16_t o[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[b][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f; // l_run: this lane's half of the keys only (merged at the end)
    // Exponents of 2: a weight is 2^(score c - m), c = scale log2 e in two floats and one rounding to f32 (the score scaled, the maximum taken off and the product with log2 e each rounded
    // left weights 2^-22 off that the bf16 terms had right).  The smaller float has the larger one's sign, so that the infinity of a key that is not seen stays one.
    constexpr float kLog2e = 0x1.715476p+0f;
    float c_hi, c_lo;
    {
        const double c = (double)a.scale * 0x1.71547652b82fep+0;
        c_hi = (float)c;
        if (fabs((double)c_hi) >= fabs(c)) c_hi = bits_to_f32(f32_to_bits(c_hi) - 1);
        c_lo = (float)(c - (double)c_hi);
    }
    const float unseen = a.scale < 0.f ? INFINITY : -INFINITY;
    const uint32_t my_last_key = prefix + qi; // causal: keys 0 .. prefix + qi
    if constexpr (GEN) {
        if (a.sinks && share == 0 && kg == 0) { // the sink's unit of mass is counted once: by half 0 of the first group of the first key split
            const float sink = bf16_to_f32(((const uint16_t*)a.sinks)[head]);
            m_run = sink * kLog2e;
            l_run = half == 0 ? (fabsf(m_run) < INFINITY ? __builtin_amdgcn_exp2f(fmaf(sink, kLog2e, -m_run)) : 1.0f) : 0.0f; // (one, but for what the maximum's rounding takes)
        }
    }
    const uint32_t query_position = suffix_position + qi;
    // heads of 256: the results stay in the accumulation registers, beside the operands in the others, and leave them in a tile that rescales them alone (left to itself the compiler
    // moves all of them every tile).  With the operands in front of the products, 2043 rows of 8 heads of 256: 77.5 -> 73.0 us; four times 1021 rows of 32 heads of 128: 99 -> 97
    auto keep = [&]() {
        if constexpr (HD > 128) {
#pragma unroll
            for (int b = 0; b < NB; ++b) asm volatile("" : "+a"(o[b]));
        }
    };

    keep();
    if (t_lo < n_tiles) {
        load_tile(t_lo);
        store_tile(t_lo & 1);
    }
    __syncthreads();
    for (uint32_t t = t_lo; t < n_tiles; ++t) {
        const int buf = t & 1;
        load_tile(t + 1 < n_tiles ? t + 1 : t); // unconditional: the compiler can count the loads in flight
        keep();
        // a wave whose queries all end before this tile has nothing to add (causal), but must keep the barriers
        const uint32_t wave_last_key = prefix + (q0 + TQ - 1 < M ? q0 + TQ - 1 : M - 1);
        const uint32_t kb = t * KEYS + kg * TK; // this group's first key
        if (wave_live && kb <= wave_last_key) {
            // ---- S^T = K Q^T
            f32x16_t sacc;
#pragma unroll
            for (int r = 0; r < 16; ++r) sacc[r] = 0.f;
            const uint8_t* kt = s_k(buf) + (kg * TK + l32) * KP + half * 16;
            // (all of a product's operands are on their way before its first instruction: read two by two, each pair was waited for)
            u32x4_t kf[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const uint4 kv = *(const uint4*)(kt + s * 32);
                kf[s] = u32x4_t{kv.x, kv.y, kv.z, kv.w};
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < NS; ++s) sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, kf[s]), __builtin_bit_cast(bf16x8_t, qf[s]), sacc, 0, 0, 0);
            // A = V^T: lane = (hd row b*32 + l32, half): keys 16 st + 4 half + {0..3} and 16 st + 8 + 4 half + {0..3}
            u32x4_t vf[2][NB];
            auto read_v = [&](int st) {
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const uint8_t* vr = s_vt(buf) + (kg * HD + b * 32 + l32) * VP + (16 * st + 4 * half) * 2;
                    const uint2 v0 = *(const uint2*)vr, v1 = *(const uint2*)(vr + 16);
                    vf[st][b] = u32x4_t{v0.x, v0.y, v1.x, v1.y};
                }
            };
            read_v(0);
            __builtin_amdgcn_sched_barrier(0);
            // ---- scale, causal mask, online softmax (lane = one query; its 16 keys: (r & 3) + 8 (r >> 2) + 4 half)
            float sc[16];
            float m_loc = -INFINITY;
            if (!GEN && kb + TK <= prefix + q0 + 1) { // every query of the wave sees the whole tile (rows past the last are nobody's)
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[r] = sacc[r];
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t key = kb + (r & 3) + 8 * (r >> 2) + 4 * half;
                    bool vis = q_live && key <= my_last_key;
                    if constexpr (GEN) { // mask.rs:31-60 on positions
                        uint32_t key_position;
                        if (key >= prefix) {
                            key_position = suffix_position + (key - prefix);
                        } else if (a.is_kv_cache_ring) {
                            key_position = prefix + key - a.ring_offset;
                            if (key_position >= prefix) key_position -= prefix;
                            vis = vis && key_position < a.ring_length;
                        } else {
                            key_position = key;
                        }
                        if (a.is_sliding_window) vis = vis && key_position <= query_position && query_position - key_position < a.sliding_window_size;
                    }
                    sc[r] = vis ? sacc[r] : unseen;
                }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) m_loc = fmaxf(m_loc, sc[r] * c_hi);
            // (A tile that raises nobody's maximum leaves the results alone: 128 products of a head of 256, and as many moves out of the accumulators and back.  A maximum that is allowed to
            // lag, so that hardly a tile rescales, was 8 us of 73 faster and is not taken: the largest weight is then no longer 1, which the two terms hold exactly, and 8 % more results
            // miss the nearest bf16.)
            m_loc = fmaxf(m_loc, other_half(m_loc));
            keep();
            if (__any(m_loc > m_run)) {
                const float m_new = fmaxf(m_run, m_loc), alpha = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m_run - m_new); // m_run = -inf => 2^-inf = 0
                l_run *= alpha, m_run = m_new;
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[b][r] *= alpha;
                keep();
            }
            const float m_ref = m_run == -INFINITY ? 0.f : m_run; // (a query that has seen no key: every score is -inf)
            float psum = 0.f;
            uint32_t p_hi[8], p_lo[8];
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[r], c_hi, fmaf(sc[r], c_lo, -m_ref))), p1 = __builtin_amdgcn_exp2f(fmaf(sc[r + 1], c_hi, fmaf(sc[r + 1], c_lo, -m_ref)));
                psum += p0 + p1;
                const float h0 = round_bf16(p0), h1 = round_bf16(p1);
                p_hi[r / 2] = pack2(h0, h1);
                p_lo[r / 2] = pack2(p0 - h0, p1 - h1);
            }
            l_run += psum;
            // ---- O^T += V^T P^T : two k16 steps (registers 0..7 and 8..15 of the score tile), P as hi + lo
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const u32x4_t ph = {p_hi[4 * st], p_hi[4 * st + 1], p_hi[4 * st + 2], p_hi[4 * st + 3]};
                const u32x4_t pl = {p_lo[4 * st], p_lo[4 * st + 1], p_lo[4 * st + 2], p_lo[4 * st + 3]};
                if (st == 0) read_v(1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int b = 0; b < NB; ++b) o[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vf[st][b]), __builtin_bit_cast(bf16x8_t, ph), o[b], 0, 0, 0);
#pragma unroll
                for (int b = 0; b < NB; ++b) o[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vf[st][b]), __builtin_bit_cast(bf16x8_t, pl), o[b], 0, 0, 0);
            }
            keep();
        }
        keep();
        if (t + 1 < n_tiles) store_tile(buf ^ 1);
        lds_barrier();
    }
    if constexpr (KG > 1) { // (every wave is past the last barrier: the stretches have been read)
        float* s_o = (float*)s_mem;
        if (kg) {
            float* mine = s_o + ((kg - 1) * 4 + wave) * PER + lane;
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
            const float* theirs = s_o + (other * 4 + wave) * PER + lane;
            const float m_o = theirs[16 * NB * 64], l_o = theirs[(16 * NB + 1) * 64], m_new = fmaxf(m_run, m_o);
            const float x = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_new), y = m_o == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_o - m_new); // (a group that saw no key: m = -inf, l = 0)
            l_run = l_run * x + l_o * y, m_run = m_new;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[b][r] = fmaf(theirs[(b * 16 + r) * 64], y, o[b][r] * x);
        }
    }
    // ---- finish: l = both halves' sums (same maximum), out[q][head][hd] = O / l
    const float l_tot = l_run + other_half(l_run);
    if (part_o) { // key split: f32 partials, row = (split, query, head)
        if (q_live) {
            const size_t row = ((size_t)share * M + qi) * a.num_heads + head;
            float* po = part_o + row * HD;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    *(float4*)(po + b * 32 + 8 * j + 4 * half) = make_float4(o[b][4 * j], o[b][4 * j + 1], o[b][4 * j + 2], o[b][4 * j + 3]);
            if (half == 0) part_ml[2 * row] = m_run, part_ml[2 * row + 1] = l_tot;
        }
        return;
    }
    if (q_live) {
        const float inv = 1.0f / l_tot;
        uint16_t* orow = out + ((size_t)qi * a.num_heads + head) * HD;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int j = 0; j < 4; ++j) { // rows (hd) 8 j + 4 half + {0..3} of block b
                uint2 w;
                w.x = pack2(o[b][4 * j] * inv, o[b][4 * j + 1] * inv);
                w.y = pack2(o[b][4 * j + 2] * inv, o[b][4 * j + 3] * inv);
                *(uint2*)(orow + b * 32 + 8 * j + 4 * half) = w;
            }
    }
}

bool attention_prefill_mfma_supported(const AttentionParams& a) {
    if (exact_mode()) return false; // reference-order mode: the scalar-order kernels of k_exact.hip
    static const uint32_t min_m = [] {
        const char* e = lab_env("UZU_ATTN_MFMA_MIN_M");
        return e ? (uint32_t)atoi(e) : 16u;
    }();
    static const bool general_on = [] { // UZU_ATTN_MFMA_GENERAL=0: sliding-window / ring / sink layers back on the VALU kernels (A/B runs)
        const char* e = lab_env("UZU_ATTN_MFMA_GENERAL");
        return !e || atoi(e) != 0;
    }();
    if (a.dt != UZU_BF16 || !a.is_causal || a.trie) return false;
    if (!general_on && (a.sinks || a.is_sliding_window || a.is_kv_cache_ring)) return false;
    if (a.is_kv_cache_ring && !a.is_sliding_window) return false; // a ring without a window does not occur (state.rs:69-136)
    if (a.suffix_length < min_m || !(a.head_dim == 64 || a.head_dim == 128 || a.head_dim == 256)) return false;
    if (a.gqa_factor == 0 || a.num_heads % a.gqa_factor) return false;
    if (a.k_head_stride % 8 || a.k_seq_stride % 8 || a.v_head_stride % 8 || a.v_seq_stride % 8) return false;
    if (!(fabsf(a.scale) >= 1e-20f && fabsf(a.scale) <= 1e20f)) return false; // (two floats of it)
    return true;
}

// out[q][head][:] = sum_s w_s O_s / sum_s w_s l_s, w_s = 2^(m_s - max m) (a split that saw no key has m = -inf, l = 0: weight 0).
// grid = rows / 4, 256 threads: 64 threads per (query, head) row, HD / 64 elements each.
// MOST: the shares that a row has at most (a body with twelve shares' loads and branches costs a launch of two shares 1.2 us of 3.4).
template <int HD, uint32_t MOST>
// gate (optional): SigmoidGate (sigmoid_gate.rs:9-22) on the merged rows in the same launch -- out = bf16(bf16(o) * sigmoid(gate)), the separate kernel's two roundings
__global__ void __launch_bounds__(256) attention_prefill_merge_kernel(const float* part_o, const float* part_ml, uint16_t* out, uint32_t rows, KeyShares shares, uint32_t tpw,
                                                                      uint32_t gqa, uint32_t heads, const uint16_t* gate) {
    constexpr int EPT = HD / 64;
    const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6), e0 = (threadIdx.x & 63) * EPT;
    if (row >= rows) return;
    const uint32_t query = row / heads, head = row - query * heads, splits = key_shares(shares, (query / TQ * gqa + head % gqa) / tpw, tpw, gqa, rows / heads, HD <= 128 ? 2 * TK : TK);
    // every share is requested before the first is used (one behind the other, a share was two trips to memory: eight shares of 517 rows 11.2 us, 9.3 so; 6.9 in a body for eight, and 14.3 for 2043 rows
    // of up to three)
    float ms[MOST], ls[MOST], po[MOST][EPT];
    uint16_t gs[EPT];
#pragma unroll
    for (uint32_t sp = 0; sp < MOST; ++sp) {
        ms[sp] = -INFINITY;
        if (sp < splits) {
            const size_t r = (size_t)sp * rows + row;
            ms[sp] = part_ml[2 * r], ls[sp] = part_ml[2 * r + 1];
#pragma unroll
            for (int e = 0; e < EPT; ++e) po[sp][e] = part_o[r * HD + e0 + e];
        }
    }
#pragma unroll
    for (int e = 0; e < EPT; ++e) gs[e] = gate ? gate[(size_t)row * HD + e0 + e] : (uint16_t)0;
    __builtin_amdgcn_sched_barrier(0);
    float m = -INFINITY;
#pragma unroll
    for (uint32_t sp = 0; sp < MOST; ++sp) m = fmaxf(m, ms[sp]);
    float acc[EPT], l = 0.f;
#pragma unroll
    for (int e = 0; e < EPT; ++e) acc[e] = 0.f;
#pragma unroll
    for (uint32_t sp = 0; sp < MOST; ++sp) {
        if (sp >= splits || ms[sp] == -INFINITY) continue;
        const float w = __builtin_amdgcn_exp2f(ms[sp] - m);
        l = fmaf(ls[sp], w, l);
#pragma unroll
        for (int e = 0; e < EPT; ++e) acc[e] = fmaf(po[sp][e], w, acc[e]);
    }
    const float inv = 1.0f / l;
    uint16_t* orow = out + (size_t)row * HD + e0;
    if (gate) {
        uint32_t bits[EPT];
#pragma unroll
        for (int e = 0; e < EPT; ++e) bits[e] = scaled_sigmoid_bf16(bf16_to_f32((uint16_t)pack2(acc[e] * inv, 0.f)), bf16_to_f32(gs[e]), kExp2fTab);
        if constexpr (EPT == 1) {
            orow[0] = (uint16_t)bits[0];
        } else {
#pragma unroll
            for (int e = 0; e < EPT; e += 2) *(uint32_t*)(orow + e) = bits[e] | (bits[e + 1] << 16);
        }
    } else if constexpr (EPT == 1) {
        orow[0] = (uint16_t)pack2(acc[0] * inv, 0.f);
    } else {
#pragma unroll
        for (int e = 0; e < EPT; e += 2) *(uint32_t*)(orow + e) = pack2(acc[e] * inv, acc[e + 1] * inv);
    }
}

// Few task groups (few kv heads x short chunks): four tasks a workgroup, which share every staged K / V tile, and the KEYS over workgroups until the chip is covered, once or twice -- or the workgroups
// thinned to one or two tasks, and no merge.  What a launch takes is estimated for each, and the least is taken.  Shares: their launch and the merge's; `stretch` us a stretch of the longest share of every
// 256 workgroups, which start the longest first; `workgroups` us per 256 of them for what they leave to the merge, and `rows` us per 10000 rows of a head that it writes.  None: the longest task, or
// the whole work at the chip's rate or the rounds' longest where those are more.  Fitted to 7600 launches, every quantum at 684 sizes (12 shapes of 64 .. 256, 40 .. 3000 rows, up to 4500 keys in front); what
// it picks is within 0.6 % of the fastest of them on the average, 4 of 684 are off by more than 10 % (20 % at the worst, 844 rows of 14 heads on 2 of 64).  Us, equal numbers of shares, one round of the
// shortest shares, and this: 32 heads on 8 of 128, 98 rows 11.9 / 12.8 / 7.3, 261 18.7 / 18.2 / 12.3, 532 24.4 / 25.9 / 20.5; 8 on 2 of 256, 831 rows 35.3 / 30.5 / 30.5, 2298 behind 2000 keys 224 / 212 /
// 195; 16 on 2 of 256, 154 behind 600 34.1 / 29.9 / 29.6.  528 sizes of eight shapes: 1.20x and 1.09x on the average.
struct PrefillPlan {
    uint32_t quantum = 0, units = 0, splits = 1; // units: workgroups a kv head
};
static uint32_t unsplit_tasks(uint32_t kv_heads, uint32_t n_tasks) { // fewer tasks per workgroup until the grid covers most of the chip
    uint32_t tpw = 4;
    while (tpw > 1 && kv_heads * ((n_tasks + tpw - 1) / tpw) < 192) tpw >>= 1;
    return tpw;
}
static PrefillPlan prefill_plan(const AttentionParams& a, uint32_t prefix, bool gated) {
    const uint32_t kv_heads = a.num_heads / a.gqa_factor, n_tasks = a.gqa_factor * ((a.suffix_length + TQ - 1) / TQ), n_groups = (n_tasks + 3) / 4, stretch = a.head_dim <= 128 ? 2 * TK : TK;
    PrefillPlan best;
    if (kv_heads * n_groups >= 192) return best;
    struct Cost {
        float none, none_stretch, shares, stretch, workgroups, rows;
    };
    const Cost us = a.head_dim == 64 ? Cost{4.0f, 1.09f, 7.6f, 1.08f, 7.8f, 2.1f} : a.head_dim == 128 ? Cost{4.6f, 1.47f, 10.6f, 1.60f, 9.9f, 1.0f} : Cost{5.3f, 2.12f, 12.3f, 2.28f, 12.6f, 3.3f};
    constexpr uint32_t kRound = kChipCus; // workgroups that the chip has at once
    const uint32_t round = std::max(1u, kRound / kv_heads);
    KeyShares shares{0, prefix};
    auto longest_of_rounds = [&](uint32_t tpw, uint64_t* all) { // the longest share of every round, added up
        uint32_t longest = 0, total = 0, in_round = 0;
        for (uint32_t y = (n_tasks + tpw - 1) / tpw; y-- > 0;) { // (as they start)
            const uint32_t length = key_stretches(shares, y, tpw, a.gqa_factor, a.suffix_length, stretch), n = key_shares(shares, y, tpw, a.gqa_factor, a.suffix_length, stretch);
            if (all) *all += length;
            for (uint32_t left = n; left;) {
                const uint32_t now = std::min(left, round - in_round);
                longest = std::max(longest, (length + n - 1) / n), left -= now, in_round += now;
                if (in_round == round) total += longest, longest = in_round = 0;
            }
        }
        return total + longest;
    };
    const uint32_t top = key_stretches(shares, n_groups - 1, 4, a.gqa_factor, a.suffix_length, stretch);
    uint64_t all = 0;
    const float rounds_none = (float)longest_of_rounds(unsplit_tasks(kv_heads, n_tasks), &all), l = (float)top, w = 1.31f * (float)(kv_heads * all) / (float)kRound;
    float least = us.none + us.none_stretch * std::max(rounds_none, sqrtf(sqrtf(l * l * l * l + w * w * w * w)));
    if (gated) least += 2.1f + 2.3e-6f * (float)a.suffix_length * (float)(a.num_heads * a.head_dim); // (the gate's own launch)
    auto plan_of = [&](uint32_t quantum) {
        shares.quantum = quantum;
        PrefillPlan p{quantum, 0, 1};
        for (uint32_t y = 0; y < n_groups; ++y) {
            const uint32_t n = key_shares(shares, y, 4, a.gqa_factor, a.suffix_length, stretch);
            p.units += n, p.splits = std::max(p.splits, n);
        }
        return p;
    };
    auto consider = [&](uint32_t quantum) {
        const PrefillPlan p = plan_of(quantum);
        if (p.splits == 1) return;
        const float t = us.shares + us.stretch * (float)longest_of_rounds(4, nullptr) + us.workgroups * (float)(kv_heads * p.units) / (float)kRound + us.rows * 1e-4f * (float)a.suffix_length * (float)a.num_heads;
        if (t < least) least = t, best = p;
    };
    for (uint32_t rounds = 1; rounds <= 2; ++rounds) { // the shortest shares that so many rounds hold (the longer the shares, the fewer workgroups)
        uint32_t low = 1, high = top;
        while (low < high) {
            const uint32_t mid = (low + high) / 2;
            if (kv_heads * plan_of(mid).units <= rounds * kRound) high = mid;
            else low = mid + 1;
        }
        consider(low);
        if (rounds == 1) consider((3 * low + 1) / 2); // (fewer, and less to merge)
    }
    return best;
}
uint32_t attention_prefill_mfma_shares(const AttentionParams& a, uint32_t prefix, bool gated) { return prefill_plan(a, prefix, gated).splits; }

uzu_status attention_prefill_mfma(hipStream_t s, const AttentionParams& a, void* out, const void* gate, uint32_t* gate_done) {
    return attention_prefill_mfma_behind(s, a, a.sequence_length > a.suffix_length ? a.sequence_length - a.suffix_length : 0, out, gate, gate_done);
}
uzu_status attention_prefill_mfma_behind(hipStream_t s, const AttentionParams& a, uint32_t prefix, void* out, const void* gate, uint32_t* gate_done) {
    if (gate_done) *gate_done = 0;
    const uint32_t kv_heads = a.num_heads / a.gqa_factor;
    const uint32_t n_tasks = a.gqa_factor * ((a.suffix_length + TQ - 1) / TQ);
    static const uint32_t force_tpw = [] {
        const char* e = lab_env("UZU_ATTN_TPW");
        return e ? (uint32_t)atoi(e) : 0u;
    }();
    static const int force_split = [] { // UZU_ATTN_KSPLIT: 1 = never split the keys (A/B runs)
        const char* e = lab_env("UZU_ATTN_KSPLIT");
        return e ? atoi(e) : 0;
    }();
    const size_t rows = (size_t)a.suffix_length * a.num_heads;
    PrefillPlan plan = force_split == 1 ? PrefillPlan{} : prefill_plan(a, prefix, gate != nullptr);
    float* part = nullptr;
    if (plan.splits > 1) part = (float*)stream_workspace(s, (size_t)plan.splits * rows * (a.head_dim + 2) * sizeof(float)); // null while a graph is being captured
    if (!part) plan = PrefillPlan{};
    const uint32_t splits = plan.splits, units = plan.units;
    const KeyShares shares{plan.quantum, prefix};
    uint32_t tpw = 4;
    if (splits == 1) {
        tpw = unsplit_tasks(kv_heads, n_tasks);
        if (force_tpw == 1 || force_tpw == 2 || force_tpw == 4) tpw = force_tpw;
    }
    const dim3 grid(kv_heads, splits > 1 ? units : (n_tasks + tpw - 1) / tpw);
    float* part_o = part;
    float* part_ml = part ? part + (size_t)splits * rows * a.head_dim : nullptr;
    const bool general = a.sinks || a.is_sliding_window || a.is_kv_cache_ring;
#define UZU_LAUNCH(H)                                                                                                                                              \
    {                                                                                                                                                              \
        UZU_PROPAGATE(launch_check([&] {                                                                                                                           \
            if (general) hipLaunchKernelGGL((attention_prefill_mfma_kernel<H, true>), grid, dim3(H <= 128 ? 512 : 256), 0, s, a, (uint16_t*)out, tpw, part_o, part_ml, shares);         \
            else hipLaunchKernelGGL((attention_prefill_mfma_kernel<H, false>), grid, dim3(H <= 128 ? 512 : 256), 0, s, a, (uint16_t*)out, tpw, part_o, part_ml, shares);                \
        }, "attention_prefill_mfma"));                                                                                                                             \
        if (!part) return UZU_OK;                                                                                                                                  \
        if (gate && gate_done) *gate_done = 1;                                                                                                                     \
        const auto merge = splits <= 2 ? attention_prefill_merge_kernel<H, 2> : splits <= 4 ? attention_prefill_merge_kernel<H, 4> : splits <= 8 ? attention_prefill_merge_kernel<H, 8> : attention_prefill_merge_kernel<H, kMaxKeySplits>; \
        return launch_check([&] { hipLaunchKernelGGL(merge, dim3((uint32_t)((rows + 3) / 4)), dim3(256), 0, s, part_o, part_ml, (uint16_t*)out, (uint32_t)rows, shares, tpw, a.gqa_factor, a.num_heads, gate_done ? (const uint16_t*)gate : nullptr); }, \
                            "attention_prefill_merge");                                                                                                            \
    }
    switch (a.head_dim) {
    case 64: UZU_LAUNCH(64);
    case 128: UZU_LAUNCH(128);
    default: UZU_LAUNCH(256);
    }
#undef UZU_LAUNCH
}

// Where the workgroups of four tasks of a full launch's sequences together cover three CUs of four, as one sequence's have to for a launch without key splits; windows, rings and sinks stay
// one by one.  (A smaller share of more than kMost sequences stays joined: 9 sequences of 120 rows, 23.8 us a layer against 15 each by themselves.)
bool attention_prefill_mfma_joins(const AttentionParams& a, uint32_t sequences) {
    if (sequences < 2 || a.sinks || a.is_sliding_window || a.is_kv_cache_ring || !attention_prefill_mfma_supported(a)) return false;
    const uint32_t n_tasks = a.gqa_factor * ((a.suffix_length + TQ - 1) / TQ);
    return sequences * (a.num_heads / a.gqa_factor) * ((n_tasks + 3) / 4) >= 192;
}
uzu_status attention_prefill_mfma_seqs(hipStream_t s, const AttentionParams& a, const AttentionSeqs& q) {
    const uint32_t n_tasks = a.gqa_factor * ((a.suffix_length + TQ - 1) / TQ);
    const dim3 grid(a.num_heads / a.gqa_factor * q.n, (n_tasks + 3) / 4);
#define UZU_LAUNCH(H)                                                                                                                                              \
    return launch_check([&] { hipLaunchKernelGGL((attention_prefill_mfma_kernel<H, false, true>), grid, dim3(H <= 128 ? 512 : 256), 0, s, a, (uint16_t*)nullptr, 4u, (float*)nullptr, (float*)nullptr, q); }, \
                        "attention_prefill_mfma_seqs")
    switch (a.head_dim) {
    case 64: UZU_LAUNCH(64);
    case 128: UZU_LAUNCH(128);
    default: UZU_LAUNCH(256);
    }
#undef UZU_LAUNCH
}

} // namespace k
} // namespace uzu
