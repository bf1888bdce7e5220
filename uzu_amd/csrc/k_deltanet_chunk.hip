// k_deltanet_chunk.hip -- DeltaNetPrefill (BU/cpu/kernel/gdn/prefill.rs:39-80) in chunked form for gfx950.
//
// The reference recurrence per value head (state S [Dv, Dk], decay a_t, write strength b_t, unit k_t, scaled q_t):
//     d_t = b_t (v_t - a_t S_{t-1} k_t)        S_t = a_t S_{t-1} + d_t k_t^T        o_t = S_t q_t
// is sequential in t, and with only Hv * Dv = 2048 independent rows a row-per-half-wave scan
// (k_deltanet.hip::delta_net_prefill_kernel) runs one wave per SIMD at ~650 cycles per token: latency, not work.
// Over a chunk of C = 32 tokens starting at S_0 the same recurrence has a closed form (A_t = prod_{i<=t} a_i):
//     (I + M) D = diag(b) (V - diag(A) K S_0^T),   M_ij = b_i (A_i / A_j) k_i.k_j   (j < i)
//     D = U - G S_0^T         (I + M) [U, G] = diag(b) [V, diag(A) K]
//     O = diag(A) Q S_0^T + P D                    P_ti = (A_t / A_i) q_t.k_i       (i <= t)
//     S_C = A_C S_0 + D^T diag(A_C / A_i) K
// U, G and P do not involve the state: `dn_chunk_prep_kernel` makes them for all chunks and heads in parallel (two 32 x 32 Gram matrices and one forward substitution with
// Dv + 128 right-hand sides each).  `dn_chunk_scan_kernel` then walks the chunks with two dependent products per chunk, G S^T and D^T K, and the outputs beside them.
// Same algebra, different rounding order: the state is no further from 64 bits than the recurrence's (dn_chunk_scan_kernel).  Decays are carried in log space
// (log 0 = -104, whose exponential is 0 in f32) so that products over a chunk cannot underflow into 0 / 0.  An infinity or a NaN would reach the whole chunk through the
// zeros of G and P, where the recurrence hands it on from its token and its value column only: the columns of a scan workgroup that meets one are walked again token by token
// (dn_recurrence_tile), by the same workgroup in the plain scan and by the fix-up in the split one.
#include <stdlib.h>

#include <type_traits>

#include "device_utils.h"
#include "internal.h"
#include "kernels.h"

namespace uzu {
namespace k {

namespace {
constexpr int CC = 32;        // tokens per chunk
constexpr int DKC = 128;      // head_k_dim
constexpr int KP = DKC + 4;   // LDS row pitch of K / Q / S rows in floats (conflict-free b128 reads across rows)
constexpr int TP = CC + 4;    // LDS row pitch of the 32 x 32 matrices (16-byte rows)
// per (chunk, value head): -G [32][128], P [32][32], A, W = A_C / A, the decays a, the strengths b; behind all of them U [32][Dv] per (chunk, value head)
constexpr int WS_P = CC * DKC, WS_A = WS_P + CC * CC, WS_W = WS_A + CC, WS_DECAY = WS_W + CC, WS_FLOATS = WS_DECAY + 2 * CC;
constexpr int SPLIT_OFF = 3 * (DKC / 16) * 4; // ScanSplit::off of a head
} // namespace

// Sequence split.  The chain of n chunk steps is the scan's whole cost (1.46 us per chunk with half of the CUs idle), and the recurrence is AFFINE in the state, row by
// row -- S_t[i,:] = S_{t-1}[i,:] a_t (I - b_t k_t k_t^T) + b_t v_t[i] k_t^T -- with the
// same linear part for every row.  So the chunks [mid, n) do not have to wait for the chunks [0, mid): they run at the same time from a ZERO state with the
// real values (Z_t, outputs Z_t q_t) and, as Dk more "value columns" per head, from the IDENTITY with zero values (H_t, outputs u_t = H_t q_t); then
//     S_t = S_mid H_t + Z_t        o_t = Z_t q_t + S_mid u_t        (S_mid = the state after chunk mid - 1)
// and `dn_chunk_fixup_kernel` adds the S_mid terms (one [tokens, Dk] x [Dk, Dv] product per head on the f32 matrix cores) before the outputs are rounded.
// Twice the scan work for segment 1, on the CUs the single chain leaves idle.  Placement decides what that buys: a segment-1 workgroup is EIGHT waves, group 0 the real tile,
// group 1 the homogeneous tile of the same head, one workgroup per CU, 2.8 us a chunk; segment 0 -- alone on its CUs at 1.46 us per chunk -- takes the larger share of the chunks.
struct ScanSplit {
    uint32_t mid_chunk; // 0: one segment (the plain scan)
    float* mid_state;   // [Hv][Dv][Dk]  final state of segment 0
    float* z_end;       // [Hv][Dv][Dk]  final state of segment 1 started from zero
    float* h_end;       // [Hv][Dk][Dk]  final homogeneous rows of segment 1 (started from the identity)
    float* o32;         // [T][Hv Dv] f32: the real tiles' own outputs (rows of segment 1: Z_t q_t; segment 0's rows are not read again)
    float* u;           // [T - 32 mid][Hv Dk] f32: H_t q_t
    uint32_t* off;      // [Hv][segment 0, segment 1, homogeneous][8 tiles][4 waves]: not 0 where a wave ends on a state value that is no number, or too large for the fix-up's products
};
static uint32_t split_mid_chunk(uint32_t n_chunks, uint32_t head_v_dim) {
    static const uint32_t min_chunks = [] { // chunks from which the scan is split (0 = never; A/B runs): the fix-up launch is 8 us + 0.12 a chunk, the shorter chain saves 0.5 a chunk
        // (17 chunks of the 0.8B model: one chain 28.6 us, split 22 + 9.9)
        const char* e = tune_env("dn_split");
        return e ? (uint32_t)atoi(e) : 24u;
    }();
    static const uint32_t pct = [] { // UZU_DN_SPLIT_PCT: segment 0's share of the chunks (its workgroups run 1.46 us per chunk, segment 1's double groups 2.8)
        const char* e = lab_env("UZU_DN_SPLIT_PCT");
        const int v = e ? atoi(e) : 66;
        return (uint32_t)(v < 10 ? 10 : v > 90 ? 90 : v);
    }();
    if (!min_chunks || n_chunks < min_chunks || head_v_dim != (uint32_t)DKC) return 0u; // (a segment-1 workgroup pairs value tile i with homogeneous tile i: Dv = Dk)
    const uint32_t mid = (n_chunks * pct + 50) / 100;
    return mid < 1 ? 1u : mid > n_chunks - 1 ? n_chunks - 1 : mid;
}
static size_t split_floats(uint32_t num_v_heads, uint32_t value_dim, uint32_t suffix_len) {
    return (size_t)2 * value_dim * DKC + (size_t)num_v_heads * DKC * DKC + (size_t)suffix_len * value_dim + (size_t)suffix_len * num_v_heads * DKC + (size_t)num_v_heads * SPLIT_OFF;
}
size_t delta_net_chunk_workspace_bytes(uint32_t num_v_heads, uint32_t value_dim, uint32_t suffix_len) {
    return ((size_t)((suffix_len + CC - 1) / CC) * ((size_t)num_v_heads * WS_FLOATS + (size_t)CC * value_dim) + split_floats(num_v_heads, value_dim, suffix_len)) * sizeof(float);
}

template <int CTRL> __device__ __forceinline__ double dpp_f64(double v) {
    const uint64_t u = f64_to_bits(v);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xF, 0xF, true), hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xF, 0xF, true);
    return bits_to_f64((uint64_t)hi << 32 | lo);
}
// log a_t, in 64 bits until an exponential of a difference is rounded: f32 prefix sums of fast decays (a = 1/e: -32 at a chunk's end) cost the state 1e-6 of its norm, the
// recurrence has 6e-8.  Decay 0: -104, whose exponential rounds to 0; a NaN or the logarithm of a negative decay stays NaN.
// The sum over the tokens up to this one, a token a lane.
__device__ __forceinline__ double log_prefix(float d, int token) {
    double l = log_wide(d);
    l = l < -104.0 ? -104.0 : l;
    // (lane i - 1, - 2, - 4, - 8 of a row of sixteen, or 0; then row 0's total to row 1)
    l += dpp_f64<0x111>(l), l += dpp_f64<0x112>(l), l += dpp_f64<0x114>(l), l += dpp_f64<0x118>(l);
    const double before = dpp_f64<0x142>(l);
    return token >= 16 ? l + before : l;
}

// grid (chunks, Hv), 256 threads.
// FUSED: DeltaNetPrefillPrep (prefill_prep.rs:30-113; k_deltanet.hip::delta_net_prefill_prep_kernel) runs inside this kernel -- the chunk's q / k rows come
// straight from the conv'd in-projection rows (bf16), are L2-normalised with that kernel's element mapping and reduction order (a wave per token, two elements per
// lane, wave_sum: the same bits), land in LDS for the Gram matrices AND in q_norm / k_norm for the scan (written by the first value head of a key head); beta and the
// decay of the chunk's tokens are computed where they are used.  Also convolving the q / k channels here (the conv kernel then rewriting the v channels only) was built,
// bit-identical, and bought nothing (9.66-9.73 vs 9.60-9.72 ms, profiles/r6_prep_fused_ab.txt): the window loads and 4 SiLUs per token cost this kernel what the conv kernel
// saved; not kept.
// What it costs is the chain of its phases, so each takes all waves or runs beside another: wave 0 the decays (three exponentials and a logarithm of a token in 64 bits) while
// the others normalise the rows, a wave's reciprocal roots all at once; the Gram tiles at and below the diagonal on the f32 matrix cores, two a wave in waves 0 and 1, one in waves 2 and 3, which make the decay
// ratios besides; the forward substitution with a thread per right-hand side, row by row as soon as the row above is known (right-looking: the sums of a row in the same order,
// the FMAs of different rows independent).  Sixteen heads of a 37-token prompt: 17.1 us (one thread a column of T, a
// sum after the other) -> 11.3, of 2043 tokens 28.6 -> 28.8 (and U and G besides).
template <bool FUSED>
__global__ void __launch_bounds__(256, 3) dn_chunk_prep_kernel(const float* q_norm, const float* k_norm, const float* beta_buf, const float* decay_buf,
                                                            float* ws, float* u_out, uint32_t num_v_heads, uint32_t num_k_heads, uint32_t head_v_dim, uint32_t key_dim, uint32_t suffix_len,
                                                            const uint16_t* in_proj, const float* a_log, const float* dt_bias, float* q_norm_out, float* k_norm_out,
                                                            uint32_t value_dim, const uint16_t* conv_rows, float* conv_state) {
    __shared__ __attribute__((aligned(16))) float sK[CC * KP], sQ[CC * KP], sV[CC * KP];
    // M (by columns) and the decay ratios: in the Q rows once the Gram products have read them (a barrier in between): 51 KB, three workgroups per CU
    float* const sMt = sQ;
    float* const sRat = sQ + CC * TP;
    static_assert(2 * CC * TP <= CC * KP, "the matrices fit in the Q rows");
    __shared__ double s_lg[CC];
    __shared__ float s_b[CC], s_ba[CC];
    __shared__ uint64_t s_exp_tab[32];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i16 = lane & 15, kq = lane >> 4;
    const uint32_t groups_per_head = num_v_heads / num_k_heads;
    const uint32_t chunk = blockIdx.x, hv = blockIdx.y, hk = hv / groups_per_head;
    const uint32_t t0 = chunk * CC;
    const uint32_t conv_dim = 2 * key_dim + value_dim;
    const size_t total_proj_dim = (size_t)conv_dim + value_dim + 2 * num_v_heads;
    float* const w_g = ws + ((size_t)chunk * num_v_heads + hv) * WS_FLOATS;
    float* const w_u = u_out + ((size_t)chunk * num_v_heads + hv) * CC * head_v_dim;
    const uint32_t live_rows = min(suffix_len - t0, (uint32_t)CC);
    auto row_of = [&](uint32_t i) { return min(i, live_rows - 1); }; // of the chunk; past the end: the last one
    // the next pass's carried conv state, the last three raw rows (T >= 3: delta_net_prefill_chunked_supported) -- the out-of-place conv kernel only reads the state; the first
    // chunk's workgroups share the channels, the first two of a thread are read here and written at the end
    auto next_state = [&](uint32_t c, float (&nx)[3]) {
#pragma unroll
        for (int tap = 0; tap < 3; ++tap) nx[tap] = bf16_to_f32(in_proj[(size_t)(suffix_len - 3 + tap) * total_proj_dim + c]);
    };
    const bool carries = FUSED && conv_state && chunk == 0;
    const uint32_t c0 = hv * 256 + tid, c_step = num_v_heads * 256;
    float nx[2][3] = {};
    if (carries) {
        if (c0 < conv_dim) next_state(c0, nx[0]);
        if (c0 + c_step < conv_dim) next_state(c0 + c_step, nx[1]);
    }
    // the chunk's values, 128 columns at a time: f32 rows in LDS
    const uint32_t v_stride = conv_rows ? conv_dim : (uint32_t)total_proj_dim;
    const uint16_t* v_base = (conv_rows ? conv_rows : in_proj) + (size_t)t0 * v_stride + 2 * key_dim + hv * head_v_dim;
    uint32_t vraw[8];
    auto load_values = [&](uint32_t column) {
        const uint16_t* v = v_base + min(column + 2 * lane, head_v_dim - 2);
#pragma unroll
        for (int r = 0; r < 8; ++r) vraw[r] = *(const uint32_t*)(v + row_of(wave + 4 * r) * v_stride);
    };
    auto put_values = [&]() {
#pragma unroll
        for (int r = 0; r < 8; ++r) *(float2*)(sV + (wave + 4 * r) * KP + 2 * lane) = make_float2(bits_to_f32(vraw[r] << 16), bits_to_f32(vraw[r] & 0xFFFF0000u));
    };
    load_values(0);
    if constexpr (FUSED) {
        if (wave) { // the rows: waves 1 .. 3, 11, 11 and 10 tokens
            const bool writer = hv % groups_per_head == 0; // one value head per key head files the rows for the scan
            constexpr int TW = 11; // every load requested before the first reduction
            uint32_t qw[TW], kw[TW];
            const int tl0 = (wave - 1) * TW, count = wave == 3 ? CC - 2 * TW : TW;
            // (conv_rows: the conv'd channels were written out of place -- k_deltanet.hip::conv_apply4_oop_kernel -- and the in-projection rows are still raw)
            const uint32_t stride = conv_rows ? conv_dim : (uint32_t)total_proj_dim;
            const uint16_t* rows = (conv_rows ? conv_rows : in_proj) + (size_t)t0 * stride + hk * DKC;
#pragma unroll
            for (int i = 0; i < TW; ++i) {
                const uint16_t* row = rows + row_of(tl0 + i) * stride;
                qw[i] = *(const uint32_t*)(row + lane * 2);
                kw[i] = *(const uint32_t*)(row + key_dim + lane * 2);
            }
            float sq = 0.f; // lane i: the square sum of token i's query, lane 16 + i: of its key
#pragma unroll
            for (int i = 0; i < TW; ++i) {
                const float qv[2] = {bits_to_f32(qw[i] << 16), bits_to_f32(qw[i] & 0xFFFF0000u)}, kv[2] = {bits_to_f32(kw[i] << 16), bits_to_f32(kw[i] & 0xFFFF0000u)};
                float q_sq = 0.f, k_sq = 0.f;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    q_sq += qv[e] * qv[e];
                    k_sq += kv[e] * kv[e];
                }
                q_sq = wave_sum(q_sq);
                k_sq = wave_sum(k_sq);
                sq = lane == i ? q_sq : lane == 16 + i ? k_sq : sq;
            }
            const float inv = 1.0f / sqrtf(sq + 1e-6f);
            const float q_scale = 1.0f / sqrtf((float)DKC);
#pragma unroll
            for (int i = 0; i < TW; ++i) {
                const uint32_t tl = tl0 + i;
                const float q_inv = bits_to_f32(__builtin_amdgcn_readlane(f32_to_bits(inv), i)), k_inv = bits_to_f32(__builtin_amdgcn_readlane(f32_to_bits(inv), 16 + i));
                float2 qn = make_float2(0.f, 0.f), kn = qn; // zero rows past the end: b = 0, a = 1 there, so they change nothing
                const bool live = tl < live_rows;
                if (live) {
                    qn = make_float2(bits_to_f32(qw[i] << 16) * q_inv * q_scale, bits_to_f32(qw[i] & 0xFFFF0000u) * q_inv * q_scale);
                    kn = make_float2(bits_to_f32(kw[i] << 16) * k_inv, bits_to_f32(kw[i] & 0xFFFF0000u) * k_inv);
                }
                if (i < count) {
                    *(float2*)(sQ + tl * KP + lane * 2) = qn;
                    *(float2*)(sK + tl * KP + lane * 2) = kn;
                    if (live && writer) {
                        *(float2*)(q_norm_out + (size_t)(t0 + tl) * key_dim + hk * DKC + lane * 2) = qn;
                        *(float2*)(k_norm_out + (size_t)(t0 + tl) * key_dim + hk * DKC + lane * 2) = kn;
                    }
                }
            }
        }
    } else {
        // K, Q rows of the chunk (zero rows past the end: b = 0, a = 1 there, so they change nothing)
        for (int idx = tid; idx < CC * (DKC / 4); idx += 256) {
            const int t = idx / (DKC / 4), c4 = idx % (DKC / 4);
            float4 kv = make_float4(0.f, 0.f, 0.f, 0.f), qv = kv;
            if (t0 + t < suffix_len) {
                kv = *(const float4*)(k_norm + (size_t)(t0 + t) * key_dim + hk * DKC + c4 * 4);
                qv = *(const float4*)(q_norm + (size_t)(t0 + t) * key_dim + hk * DKC + c4 * 4);
            }
            *(float4*)(sK + t * KP + c4 * 4) = kv;
            *(float4*)(sQ + t * KP + c4 * 4) = qv;
        }
    }
    if (wave == 0) { // decays and strengths, a token a lane
        const uint32_t tok = t0 + row_of(lane);
        float raw_b, raw_a;
        if constexpr (FUSED) {
            const uint16_t* row = in_proj + (size_t)tok * total_proj_dim + conv_dim + value_dim;
            raw_b = bf16_to_f32(row[hv]), raw_a = bf16_to_f32(row[num_v_heads + hv]);
        } else raw_b = beta_buf[(size_t)tok * num_v_heads + hv], raw_a = decay_buf[(size_t)tok * num_v_heads + hv];
        if (lane < 32) s_exp_tab[lane] = kExp2fTab[lane];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // (this wave reads it now, the others behind the barrier)
        if (lane < CC) {
            float d = 1.0f, b = 0.0f;
            if ((uint32_t)lane < live_rows) {
                if constexpr (FUSED) {
                    b = 1.0f / (1.0f + expf_glibc_tab(-raw_b, s_exp_tab));
                    const float sp_in = raw_a + dt_bias[hv];
                    const float sp = sp_in > 20.0f ? sp_in : logf_glibc(1.0f + expf_glibc_tab(sp_in, s_exp_tab));
                    const float log_decay = -expf_glibc_tab(a_log[hv], s_exp_tab) * sp;
                    d = expf_glibc_tab(log_decay, s_exp_tab);
                } else d = raw_a, b = raw_b;
            }
            const double lg = log_prefix(d, lane);
            const float a_t = exp_wide(lg, s_exp_tab);
            s_lg[lane] = lg, s_b[lane] = b, s_ba[lane] = -b * a_t;
            w_g[WS_DECAY + lane] = d, w_g[WS_DECAY + CC + lane] = b;
            w_g[WS_A + lane] = a_t;
        }
    }
    put_values();
    __syncthreads();
    // Gram tiles (rows 16 x .., columns 16 y ..; D: rows 4 kq + r, column i16): waves 0, 1: K K^T (0, 0) and (1, 0) | (1, 1), Q K^T (0, 0); waves 2, 3: Q K^T (1, 0) | (1, 1)
    typedef __attribute__((ext_vector_type(4))) float acc_t;
    auto gram = [&](const float* rows, int x, int y) {
        const float *xr = rows + (16 * x + i16) * KP + 4 * kq, *yr = sK + (16 * y + i16) * KP + 4 * kq;
        acc_t part[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int g = 0; g < DKC / 16; ++g) { // contraction index of step e in quarter kq: 16 g + 4 kq + e
            const f32x4_v a = *(const f32x4_v*)(xr + 16 * g), b = *(const f32x4_v*)(yr + 16 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) part[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], part[e & 1], 0, 0, 0);
        }
        return part[0] + part[1];
    };
    acc_t tile0, tile1 = {0.f, 0.f, 0.f, 0.f};
    if (wave == 0) tile0 = gram(sK, 0, 0), tile1 = gram(sK, 1, 0);
    else if (wave == 1) tile0 = gram(sK, 1, 1), tile1 = gram(sQ, 0, 0);
    else tile0 = gram(sQ, 1, wave - 2);
    float ratio[5];
    if (wave >= 2) { // A_i / A_j for j <= i: 528 of them, row r and row 31 - r together 33
#pragma unroll
        for (int n = 0; n < 5; ++n) {
            const int p = min(tid - DKC + 128 * n, 527), r = p / 33, q = p % 33, i = q <= r ? r : 31 - r, j = q <= r ? q : q - r - 1;
            ratio[n] = exp_wide(s_lg[i] - s_lg[j], s_exp_tab);
        }
    }
    __syncthreads(); // every wave has read its K / Q rows: the Q rows become the matrices
    if (wave >= 2) {
#pragma unroll
        for (int n = 0; n < 5; ++n) {
            const int p = min(tid - DKC + 128 * n, 527), r = p / 33, q = p % 33, i = q <= r ? r : 31 - r, j = q <= r ? q : q - r - 1;
            sRat[i * TP + j] = ratio[n];
        }
    }
    __syncthreads();
    auto put_m = [&](const acc_t& kk, int x, int y) { // M_ij = b_i A_i / A_j k_i.k_j below the diagonal, by columns
        const int j = 16 * y + i16, i0 = 16 * x + 4 * kq;
        f32x4_v m;
#pragma unroll
        for (int r = 0; r < 4; ++r) m[r] = j < i0 + r ? s_b[i0 + r] * sRat[(i0 + r) * TP + j] * kk[r] : 0.0f;
        *(f32x4_v*)(sMt + j * TP + i0) = m;
    };
    auto put_p = [&](const acc_t& qk, int x, int y) {
        const int j = 16 * y + i16, i0 = 16 * x + 4 * kq;
#pragma unroll
        for (int r = 0; r < 4; ++r) w_g[WS_P + (i0 + r) * CC + j] = j <= i0 + r ? sRat[(i0 + r) * TP + j] * qk[r] : 0.0f;
    };
    if (tid < CC) { // behind a column of M: its row's coefficients of the right-hand sides
        w_g[WS_W + tid] = exp_wide(s_lg[CC - 1] - s_lg[tid], s_exp_tab); // A_C / A_t
        *(float2*)(sMt + tid * TP + CC) = make_float2(s_b[tid], s_ba[tid]);
    }
    if (wave == 0) put_m(tile0, 0, 0), put_m(tile1, 1, 0);
    else if (wave == 1) put_m(tile0, 1, 1), put_p(tile1, 0, 0);
    else {
        put_p(tile0, 1, wave - 2);
        if (wave == 2) { // P above the diagonal
#pragma unroll
            for (int r = 0; r < 4; ++r) w_g[WS_P + (4 * kq + r) * CC + 16 + i16] = 0.0f;
        }
    }
    __syncthreads();
    // (I + M) X = diag(b) [-diag(A) K, V]: column c of 128 + Dv in a thread.  A row's sum over the rows above it is gathered first, its own term joins it in one rounding: started
    // from that term, which is the larger one, the sum would be rounded at its size 31 times (a state of fast decays 1.6 times as far from 64 bits)
    const bool key = tid < DKC; // (a whole wave's columns)
    for (uint32_t v0 = 0; v0 < head_v_dim; v0 += DKC) {
        const uint32_t c = key ? tid : v0 + tid - DKC;
        if (v0) { // values wider than 128
            __syncthreads();
            load_values(v0);
            put_values();
            __syncthreads();
        }
        if (key ? v0 != 0 : c >= head_v_dim) continue;
        const float* val = key ? sK + tid : sV + tid - DKC;
        float x[CC] = {};
        f32x4_v m[2][8]; // column j of M, the next one on its way
        float2 coef[2];
        float rhs[2];
        auto column = [&](int j) {
            coef[j & 1] = *(const float2*)(sMt + j * TP + CC);
            rhs[j & 1] = val[j * KP];
#pragma unroll
            for (int q = (j + 1) / 4; q < 8; ++q) m[j & 1][q] = *(const f32x4_v*)(sMt + j * TP + 4 * q);
        };
        column(0);
#pragma unroll
        for (int j = 0; j < CC; ++j) {
            if (j + 1 < CC) column(j + 1);
            x[j] = fmaf(key ? coef[j & 1].y : coef[j & 1].x, rhs[j & 1], -x[j]);
#pragma unroll
            for (int i = j + 1; i < CC; ++i) x[i] = fmaf(m[j & 1][i / 4][i % 4], x[j], x[i]);
            __builtin_amdgcn_sched_barrier(0); // (all columns at once would not fit the registers)
        }
        float* dst = key ? w_g + c : w_u + c;
        const uint32_t stride = key ? (uint32_t)DKC : head_v_dim;
#pragma unroll
        for (int i = 0; i < CC; ++i) dst[(size_t)i * stride] = x[i];
    }
    if (carries) {
#pragma unroll
        for (int tap = 0; tap < 3; ++tap) {
            if (c0 < conv_dim) conv_state[(size_t)c0 * 3 + tap] = nx[0][tap];
            if (c0 + c_step < conv_dim) conv_state[(size_t)(c0 + c_step) * 3 + tap] = nx[1][tap];
        }
        for (uint32_t c = c0 + 2 * c_step; c < conv_dim; c += c_step) {
            next_state(c, nx[0]);
#pragma unroll
            for (int tap = 0; tap < 3; ++tap) conv_state[(size_t)c * 3 + tap] = nx[0][tap];
        }
    }
}

// The recurrence token by token from the state in memory: value columns [dv_base, dv_base + 16) of head hv, 256 threads, 16 lanes a column.
// (v_row_stride != 0: `in_proj` is the out-of-place conv buffer, rows of conv_dim channels in the same q | k | v order)
__device__ __forceinline__ void dn_recurrence_tile(const float* q_norm, const float* k_norm, const uint16_t* in_proj, const float* ws, float* state, uint16_t* out, uint32_t hv, uint32_t dv_base,
                                                uint32_t num_v_heads, uint32_t num_k_heads, uint32_t head_v_dim, uint32_t key_dim, uint32_t value_dim, uint32_t suffix_len, uint32_t v_row_stride) {
    const size_t v_stride = v_row_stride ? (size_t)v_row_stride : (size_t)2 * key_dim + 2 * value_dim + 2 * num_v_heads;
    const uint32_t hk = hv / (num_v_heads / num_k_heads), col = threadIdx.x >> 4, part = threadIdx.x & 15;
    float* srow = state + ((size_t)hv * head_v_dim + dv_base + col) * DKC + 8 * part;
    float sv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) sv[e] = srow[e];
    for (uint32_t t = 0; t < suffix_len; ++t) {
        const float* w = ws + ((size_t)(t / CC) * num_v_heads + hv) * WS_FLOATS + WS_DECAY + t % CC;
        const float *kr = k_norm + (size_t)t * key_dim + hk * DKC + 8 * part, *qr = q_norm + (size_t)t * key_dim + hk * DKC + 8 * part;
        const float a = w[0], b = w[CC], v = bf16_to_f32(in_proj[(size_t)t * v_stride + 2 * key_dim + hv * head_v_dim + dv_base + col]);
        float sk = 0.f, o = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) sk = fmaf(sv[e], kr[e], sk);
        const float d = b * (v - a * group_sum<16>(sk));
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            sv[e] = a * sv[e] + d * kr[e];
            o = fmaf(sv[e], qr[e], o);
        }
        o = group_sum<16>(o);
        if (part == 0) out[(size_t)t * value_dim + hv * head_v_dim + dv_base + col] = f32_to_bf16(o);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) srow[e] = sv[e];
}

// The scan, v_mfma_f32_16x16x4_f32 throughout -- f32 operands, exact f32 products, f32 accumulation.  Four waves own 16 value columns of a head:
//   stage 1  waves 0, 1: D = U - G S^T for 16 tokens each, 32 MFMAs; waves 2, 3: Q S^T
//   stage 2  S = A_C S + (D W)^T K   every wave owns 32 dk of the state in its accumulators, 2 x 8 MFMAs
//   stage 3  O = A Q S^T + P D   waves 2, 3: 8 MFMAs, behind their part of the new state
// The chunk chain is the cost, so nothing else is on it: every operand but the state and D goes from memory straight into the registers that the MFMAs read, one chunk ahead
// (G, U, P as the preparation wrote them, Q and K as rows); only S and D pass through LDS, with a barrier each.  (K, Q, T and P staged in LDS, T as a third dependent product,
// four barriers: 2.75 us a chunk; this form 1.46, a segment-1 workgroup of two tiles 2.8.)
// MFMA operand layout (16x16x4): A lane l = row l % 16, k-quarter l / 16; B lane l = column l % 16, k-quarter l / 16; C / D four
// registers = rows 4 (l / 16) + r of column l % 16.  Contraction index of step (g, e) in quarter q: stage 1 dk = 16 g + 4 q + e, stage 3 token 8 q + s (a lane's values
// lie together in memory); stage 2 token 4 s + q: the products are added in time order and the late tokens, which weigh most under a decay, come last.  With that, four
// chains in stage 1 and the old state added behind the chunk's own products, the state of 16 to 200 tokens is 0.4 to 1.0 times as far from 64 bits as the recurrence token by token.
//
// DUAL (ScanSplit): grid (2 Dv / 16, Hv), 512 threads = two such groups of four waves;
//   workgroups [0, Dv / 16) of a head: segment 0, chunks [0, mid): group 0 = the value tile from the carried state; group 1 leaves;
//   the others:                        segment 1, chunks [mid, n): group 0 = the value tile from a zero state, group 1 = the homogeneous tile (identity, U = 0).
template <bool DUAL>
__global__ void __launch_bounds__(DUAL ? 512 : 256) dn_chunk_scan_kernel(const float* q_norm, const float* k_norm, const uint16_t* in_proj, const float* ws, const float* u_ws, const float* state_in,
                                                                         float* state, uint16_t* out, uint32_t num_v_heads, uint32_t num_k_heads, uint32_t head_v_dim, uint32_t key_dim,
                                                                         uint32_t value_dim, uint32_t suffix_len, ScanSplit sp, uint32_t v_row_stride) {
    constexpr int DVT = 16, DP = CC + 4; // value columns of a tile; LDS pitch of D's columns
    __shared__ __attribute__((aligned(16))) float smem[DUAL ? 2 : 1][DVT * KP + 2 * DVT * DP];
    __shared__ uint32_t s_off[4];
    const int tid = threadIdx.x, grp = DUAL ? __builtin_amdgcn_readfirstlane(tid >> 8) : 0, ltid = tid & 255, lane = ltid & 63, wave = __builtin_amdgcn_readfirstlane(ltid >> 6), i16 = lane & 15, kq = lane >> 4;
    float* const sS = smem[grp];           // [DVT][KP]: the state's rows (value columns)
    float* const sD = sS + DVT * KP;       // [DVT][DP]: D by value columns, tokens in order
    float* const sDw = sD + DVT * DP;      // D W, token 4 s + q at 8 q + s
    // XCD-aware (head, value tile) <- workgroup: consecutive workgroup ids go round the 8 XCDs, and the workgroups of a head all walk
    // the head's K / Q / G rows: with the plain (x = tile, y = head) numbering every one of them sits on another XCD and the rows are fetched
    // 8 times.  Here XCD x takes the pairs [x * total / 8, (x + 1) * total / 8): a head's tiles share one L2.
    uint32_t hv = blockIdx.y, tile = blockIdx.x;
    {
        const uint32_t nx = gridDim.x, total = nx * gridDim.y, lin = blockIdx.x + nx * blockIdx.y;
        if (total % 8 == 0) {
            const uint32_t pair = (lin % 8) * (total / 8) + lin / 8;
            hv = pair / nx, tile = pair % nx;
        }
    }
    const uint32_t tiles_v = head_v_dim / DVT;
    const bool seg1 = DUAL && tile >= tiles_v, homog = seg1 && grp == 1;
    if (DUAL && !seg1 && grp == 1) return; // (whole waves, in front of every barrier)
    if (seg1) tile -= tiles_v;
    const uint32_t dv_base = tile * DVT, hk = hv / (num_v_heads / num_k_heads);
    const uint32_t n_chunks = (suffix_len + CC - 1) / CC;
    const uint32_t c_begin = seg1 ? sp.mid_chunk : 0u, c_end = DUAL && !seg1 ? sp.mid_chunk : n_chunks;

    // the state: wave w owns dk 32 w .. in accumulator layout, creg[t][r] = S[dv = 4 kq + r][dk = 32 w + 2 i16 + t]
    f32x4_v creg[2];
    const size_t s_at = ((size_t)hv * head_v_dim + dv_base + 4 * kq) * DKC + 32 * wave + 2 * i16;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float2 v = make_float2(0.f, 0.f);
        if (!seg1) v = *(const float2*)(state_in + s_at + (size_t)r * DKC);
        else if (homog) {
            const uint32_t one = dv_base + 4 * kq + r, dk = 32 * wave + 2 * i16;
            v = make_float2(one == dk ? 1.f : 0.f, one == dk + 1 ? 1.f : 0.f);
        }
        creg[0][r] = v.x, creg[1][r] = v.y;
    }
    auto publish = [&]() {
#pragma unroll
        for (int r = 0; r < 4; ++r) *(float2*)(sS + (4 * kq + r) * KP + 32 * wave + 2 * i16) = make_float2(creg[0][r], creg[1][r]);
    };

    auto mfma4 = [](float a, float b, f32x4_v c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); };
    float off_sum = 0.f; // plain scan: 0, or NaN behind an output or a state value that is no number
    const int tb = 16 * (wave & 1);
    const uint32_t u_keep = homog ? 0u : 0xFFFFFFFFu;
    // segment 0's outputs (and the plain scan's) are final; segment 1's go to f32 rows that the fix-up finishes
    uint16_t* const out16 = out + (size_t)hv * head_v_dim + dv_base + i16;
    const size_t o_stride = homog ? (size_t)num_v_heads * DKC : (size_t)value_dim;
    float* const o32 = !DUAL ? nullptr : homog ? sp.u + (size_t)hv * DKC + dv_base + i16 - (size_t)sp.mid_chunk * CC * o_stride : sp.o32 + (size_t)hv * head_v_dim + dv_base + i16;

    // The chain, once for the waves of each role: a role's or a lane's condition around loads or stores of the loop makes the compiler wait, at the join, for the chunk's stores and the
    // next chunk's operands with them (3.2 us a chunk).  Only the last chunk can be ragged.
    auto walk = [&](auto front_c, auto seg1_c) {
        constexpr bool FRONT = decltype(front_c)::value, SEG1 = decltype(seg1_c)::value; // stage 1: D or Q S^T
        struct Operands {
            f32x4_v x[8], p[2], aw;
            float u[4], a_c;
            float2 k[8];
        };
        // one chunk's operands, piece by piece.  WHOLE: the chunk has all its tokens (uniform bases, the lane's offset); else rows past the end are the last one (G and U are zero there,
        // outputs are not stored)
        const uint32_t x_lane = FRONT ? (uint32_t)((tb + i16) * DKC + 4 * kq) : (uint32_t)(tb + i16) * key_dim + 4 * kq, k_lane = (uint32_t)kq * key_dim + 32 * wave + 2 * i16;
        auto block = [&](uint32_t c) { return ws + ((size_t)c * num_v_heads + hv) * WS_FLOATS; };
        auto fetch_x = [&](uint32_t c, Operands& o, int g, auto whole) {
            if constexpr (FRONT) o.x[g] = *(const f32x4_v*)(block(c) + x_lane + 16 * g);
            else if constexpr (decltype(whole)::value) o.x[g] = *(const f32x4_v*)(q_norm + (size_t)c * CC * key_dim + hk * DKC + x_lane + 16 * g);
            else o.x[g] = *(const f32x4_v*)(q_norm + (size_t)min(c * CC + tb + i16, suffix_len - 1) * key_dim + hk * DKC + 4 * kq + 16 * g);
        };
        auto fetch_k = [&](uint32_t c, Operands& o, int s2, auto whole) {
            if constexpr (decltype(whole)::value) o.k[s2] = *(const float2*)(k_norm + (size_t)(c * CC + 4 * s2) * key_dim + hk * DKC + k_lane);
            else o.k[s2] = *(const float2*)(k_norm + (size_t)min(c * CC + 4 * s2 + kq, suffix_len - 1) * key_dim + hk * DKC + 32 * wave + 2 * i16);
        };
        auto fetch_rest = [&](uint32_t c, Operands& o) {
            const float* w = block(c);
            if constexpr (FRONT) {
                const float* ur = u_ws + ((size_t)c * num_v_heads + hv) * CC * head_v_dim + (uint32_t)((tb + 4 * kq) * head_v_dim + dv_base + i16);
#pragma unroll
                for (int r = 0; r < 4; ++r) o.u[r] = ur[r * head_v_dim];
            } else {
                const float* pr = w + WS_P + (uint32_t)((tb + i16) * CC + 8 * kq);
                o.p[0] = *(const f32x4_v*)pr, o.p[1] = *(const f32x4_v*)(pr + 4);
            }
            o.aw = *(const f32x4_v*)(w + (FRONT ? WS_W : WS_A) + (uint32_t)(tb + 4 * kq));
            o.a_c = w[WS_A + CC - 1];
        };
        auto step_barrier = [&]() { // (waves 2, 3 write nothing in front of the first one: their MFMAs would be moved behind it, after those that they are to run beside)
            __builtin_amdgcn_sched_barrier(0);
            lds_barrier();
            __builtin_amdgcn_sched_barrier(0);
        };
        // The next chunk's operands are requested one by one between the MFMAs: 24 requests in a row keep a wave from its first MFMA until the L1 has served them (2.2 us a chunk
        // instead of 1.46)
        auto step = [&](uint32_t c, const Operands& o, Operands& next, bool ragged, auto whole) {
            const uint32_t n = c + 1 < c_end ? c + 1 : c; // unconditional (the last chunk refetches itself)
            // ---- stage 1
            f32x4_v part[4] = {}; // (four chains: shorter, and nearer to the exact sum than one)
            const float* sr = sS + i16 * KP + 4 * kq;
            f32x4_v sb[8];
#pragma unroll
            for (int g = 0; g < 8; ++g) sb[g] = *(const f32x4_v*)(sr + 16 * g);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < 8; ++g) {
                fetch_x(n, next, g, whole);
#pragma unroll
                for (int e = 0; e < 4; ++e) part[e] = mfma4(o.x[g][e], sb[g][e], part[e]);
                __builtin_amdgcn_sched_barrier(0);
            }
            f32x4_v acc = (part[0] + part[1]) + (part[2] + part[3]);
            if constexpr (FRONT) {
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[r] += bits_to_f32(f32_to_bits(o.u[r]) & u_keep); // (last: U is the larger term, and in front of the chain it would be rounded eight times)
                *(f32x4_v*)(sD + i16 * DP + tb + 4 * kq) = acc;
#pragma unroll
                for (int r = 0; r < 4; ++r) sDw[i16 * DP + 8 * r + tb / 4 + kq] = acc[r] * o.aw[r];
            }
            step_barrier();
            // ---- stage 2
            const f32x4_v d0 = *(const f32x4_v*)(sDw + i16 * DP + 8 * kq), d1 = *(const f32x4_v*)(sDw + i16 * DP + 8 * kq + 4); // A operand: row = value column i16
            f32x4_v u[2] = {};
#pragma unroll
            for (int s2 = 0; s2 < 8; ++s2) {
                const float d = s2 < 4 ? d0[s2 & 3] : d1[s2 & 3];
                fetch_k(n, next, s2, whole);
                u[0] = mfma4(d, o.k[s2].x, u[0]), u[1] = mfma4(d, o.k[s2].y, u[1]);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) creg[t][r] = fmaf(creg[t][r], o.a_c, u[t][r]);
            publish(); // (every wave has read the old state: the barrier above)
            __builtin_amdgcn_sched_barrier(0);
            fetch_rest(n, next);
            // ---- stage 3
            if constexpr (!FRONT) {
                const f32x4_v e0 = *(const f32x4_v*)(sD + i16 * DP + 8 * kq), e1 = *(const f32x4_v*)(sD + i16 * DP + 8 * kq + 4);
                f32x4_v y = o.aw * acc;
#pragma unroll
                for (int s2 = 0; s2 < 8; ++s2) y = mfma4(o.p[s2 >> 2][s2 & 3], s2 < 4 ? e0[s2 & 3] : e1[s2 & 3], y);
                const uint32_t t = c * CC + tb + 4 * kq;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (ragged && t + r >= suffix_len) continue;
                    if constexpr (SEG1) o32[(size_t)(t + r) * o_stride] = y[r];
                    else out16[(size_t)(t + r) * value_dim] = f32_to_bf16(y[r]);
                    if constexpr (!DUAL) off_sum = fmaf(y[r], 0.f, off_sum);
                }
            }
            step_barrier();
        };
        typedef std::integral_constant<bool, true> yes;
        typedef std::integral_constant<bool, false> no;
        Operands even, odd;
#pragma unroll
        for (int g = 0; g < 8; ++g) fetch_x(c_begin, even, g, no());
#pragma unroll
        for (int s2 = 0; s2 < 8; ++s2) fetch_k(c_begin, even, s2, no());
        fetch_rest(c_begin, even);
        publish();
        lds_barrier();
        const uint32_t full = min(c_end, suffix_len / CC); // chunks [c_begin, full) have all their tokens
        uint32_t c = c_begin;
        for (; c + 2 < full; c += 2) step(c, even, odd, false, yes()), step(c + 1, odd, even, false, yes());
        for (; c < c_end; ++c) { // at most three
            step(c, even, odd, c >= full, no());
            even = odd;
        }
    };
    typedef std::integral_constant<bool, true> yes;
    typedef std::integral_constant<bool, false> no;
    if (DUAL && seg1) {
        if (wave < 2) walk(yes(), std::integral_constant<bool, DUAL>());
        else walk(no(), std::integral_constant<bool, DUAL>());
    } else if (wave < 2) walk(yes(), no());
    else walk(no(), no());
    if constexpr (DUAL) {
        // (whatever of a chunk is no number, but for a query, which its own outputs alone see, makes a row of D none, and D stays in the state: 0 times it is none either)
        uint32_t peak = 0; // the largest magnitude's bits; a NaN's are larger than any
        float* sfin = homog ? sp.h_end + ((size_t)hv * DKC + dv_base + 4 * kq) * DKC + 32 * wave + 2 * i16 : (seg1 ? sp.z_end : sp.mid_state) + s_at;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            *(float2*)(sfin + (size_t)r * DKC) = make_float2(creg[0][r], creg[1][r]);
            peak = max(peak, max(f32_to_bits(creg[0][r]) & 0x7FFFFFFFu, f32_to_bits(creg[1][r]) & 0x7FFFFFFFu));
        }
        const bool off = __ballot(peak > f32_to_bits(0x1p60f)) != 0; // (128 products of two numbers up to that are a number)
        if (lane == 0) sp.off[((hv * 3 + (homog ? 2 : seg1 ? 1 : 0)) * (DKC / 16) + dv_base / 16) * 4 + wave] = off;
        return;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) off_sum = fmaf(creg[t][r], 0.f, off_sum);
    const bool off = __ballot(!(off_sum == 0.f)) != 0;
    if (lane == 0) s_off[wave] = off;
    lds_barrier();
    if (s_off[0] | s_off[1] | s_off[2] | s_off[3]) {
        __syncthreads(); // (every wave's own outputs have been written: those below replace them)
        dn_recurrence_tile(q_norm, k_norm, in_proj, ws, state, out, hv, dv_base, num_v_heads, num_k_heads, head_v_dim, key_dim, value_dim, suffix_len, v_row_stride);
        return;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) *(float2*)(state + s_at + (size_t)r * DKC) = make_float2(creg[0][r], creg[1][r]);
}

// The S_mid terms of a split scan (see ScanSplit).  grid (tok_blocks + Dk / 16, Hv), 4 waves;
// v_mfma_f32_16x16x4_f32 with the operand layout of the scan (lane l: row / column l % 16, contraction indices 32 (l / 16) + s over 32 steps: a lane's
// 32 operand values are consecutive in memory).  Dv = Dk = 128 (split_mid_chunk).
//   the first tok_blocks:    64 tokens of segment 1:   out[t, dv] = bf16(o32[t, dv] + sum_dk u[t, dk] S_mid[dv, dk])    wave w = tokens 16 w ..: A = its u rows,
//                                                      B = S_mid rows from LDS (the head's state staged once per workgroup: one global round trip in all)
//   the last Dk / 16 blocks: 16 state columns:         S[dv, dk] = z_end[dv, dk] + sum_j S_mid[dv, j] h_end[j, dk]       A = S_mid rows, B = h_end columns
constexpr int FIX_TOK = 64;
constexpr size_t kFixLdsBytes = (size_t)DKC * KP * sizeof(float); // S_mid of one head, rows 4 banks apart
// Value tiles that ScanSplit::off names are left alone, and block i of the last ones walks tile i token by token instead: the state in memory is still the one before the pass there.
__global__ void __launch_bounds__(256) dn_chunk_fixup_kernel(ScanSplit sp, float* state, uint16_t* out, uint32_t num_v_heads, uint32_t head_v_dim, uint32_t value_dim, uint32_t suffix_len,
                                                             const float* q_norm, const float* k_norm, const uint16_t* in_proj, const float* ws, uint32_t num_k_heads, uint32_t key_dim,
                                                             uint32_t v_row_stride) {
    constexpr uint32_t DV_TILES = DKC / 16;
    extern __shared__ __attribute__((aligned(16))) float fix_smem[]; // [Dv][KP]: S_mid of the head (token blocks)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i16 = lane & 15, kq = lane >> 4;
    const uint32_t hv = blockIdx.y, t_mid = sp.mid_chunk * CC, T2 = suffix_len - t_mid;
    const uint32_t tok_blocks = (T2 + FIX_TOK - 1) / FIX_TOK;
    const float* smid = sp.mid_state + (size_t)hv * head_v_dim * DKC;
    uint4 off4 = make_uint4(0, 0, 0, 0);
    if (lane < 3 * (int)DV_TILES) off4 = *(const uint4*)(sp.off + (size_t)hv * SPLIT_OFF + 4 * lane);
    auto off_tiles = [&]() -> uint32_t { // (a homogeneous tile serves every value tile)
        const uint64_t b = __ballot((off4.x | off4.y | off4.z | off4.w) != 0);
        return b >> (2 * DV_TILES) ? (1u << DV_TILES) - 1 : (uint32_t)(b | b >> DV_TILES) & ((1u << DV_TILES) - 1);
    };
    auto mfma4 = [](float a, float b, f32x4_v c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); };
    // the token blocks come first in the grid: they are the long ones (one global round trip + 256 matrix instructions per wave)
    if (blockIdx.x < tok_blocks) {
        // every global operand is requested before anything is consumed: S_mid (16 x 16 bytes per thread, through LDS), this wave's u rows, its o32 values
        f32x4_v sm[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) sm[r] = *(const f32x4_v*)(smid + (size_t)(tid + 256 * r) * 4);
        const uint32_t tok = blockIdx.x * FIX_TOK + 16 * wave; // this wave's 16 tokens, relative to segment 1 (past the end: computed on clamped rows, never stored)
        const size_t u_stride = (size_t)num_v_heads * DKC;
        const uint32_t row = min(tok + (uint32_t)i16, T2 - 1); // A: row = token
        const float* ur = sp.u + (size_t)row * u_stride + hv * DKC + 32 * kq;
        f32x4_v ua[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) ua[q] = *(const f32x4_v*)(ur + 4 * q);
        float prev[DV_TILES][4]; // this lane's o32 values: rows 4 kq + r, column 16 vt + i16
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t t = min(tok + 4 * kq + r, T2 - 1);
            const float* pr = sp.o32 + (size_t)(t_mid + t) * value_dim + (size_t)hv * head_v_dim + i16;
#pragma unroll
            for (uint32_t vt = 0; vt < DV_TILES; ++vt) prev[vt][r] = pr[vt * 16];
        }
        __builtin_amdgcn_sched_barrier(0); // (every request is out before the first wait)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t e = (tid + 256 * r) * 4; // element of the [Dv][Dk] state
            *(f32x4_v*)(fix_smem + (e / DKC) * KP + e % DKC) = sm[r];
        }
        const uint32_t skip = off_tiles();
        lds_barrier();
#pragma unroll
        for (uint32_t vt = 0; vt < DV_TILES; ++vt) {
            const float* br = fix_smem + (vt * 16 + i16) * KP + 32 * kq; // B: column dv = 16 vt + i16
            f32x4_v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const f32x4_v b = *(const f32x4_v*)(br + 4 * q);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc = mfma4(ua[q][e], b[e], acc);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) { // rows = tokens 4 kq + r of the tile, column = dv
                const uint32_t t = tok + 4 * kq + r;
                if (t < T2 && !(skip >> vt & 1)) out[(size_t)(t_mid + t) * value_dim + (size_t)hv * head_v_dim + vt * 16 + i16] = f32_to_bf16(prev[vt][r] + acc[r]);
            }
        }
    } else {
        const uint32_t dk0 = (blockIdx.x - tok_blocks) * 16;
        const float* hend = sp.h_end + (size_t)hv * DKC * DKC;
        float hb[32]; // B: column dk = dk0 + i16, contraction index j = 32 kq + s
#pragma unroll
        for (int s2 = 0; s2 < 32; ++s2) hb[s2] = hend[(size_t)(32 * kq + s2) * DKC + dk0 + i16];
        // this wave's two value tiles (wave, wave + 4): all of their S_mid rows and z_end values are requested before the first product (read in place, every
        // 16-byte operand was a round trip of its own in front of four matrix instructions)
        f32x4_v sa[2][8];
        float zv[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t vt = wave + 4 * h;
            const float* ar = smid + (size_t)(vt * 16 + i16) * DKC + 32 * kq; // A: row dv = 16 vt + i16
#pragma unroll
            for (int q = 0; q < 8; ++q) sa[h][q] = *(const f32x4_v*)(ar + 4 * q);
#pragma unroll
            for (int r = 0; r < 4; ++r) zv[h][r] = sp.z_end[((size_t)hv * head_v_dim + vt * 16 + 4 * kq + r) * DKC + dk0 + i16];
        }
        __builtin_amdgcn_sched_barrier(0); // (the scheduler would sink the loads back to their uses)
        const uint32_t skip = off_tiles();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t vt = wave + 4 * h;
            f32x4_v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 8; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc = mfma4(sa[h][q][e], hb[4 * q + e], acc);
#pragma unroll
            for (int r = 0; r < 4; ++r) // rows dv = 16 vt + 4 kq + r, column dk
                if (!(skip >> vt & 1)) state[((size_t)hv * head_v_dim + vt * 16 + 4 * kq + r) * DKC + dk0 + i16] = zv[h][r] + acc[r];
        }
        const uint32_t tile = blockIdx.x - tok_blocks;
        if (skip >> tile & 1) dn_recurrence_tile(q_norm, k_norm, in_proj, ws, state, out, hv, tile * 16, num_v_heads, num_k_heads, head_v_dim, key_dim, value_dim, suffix_len, v_row_stride);
    }
}

bool delta_net_prefill_chunked_supported(uint32_t num_v_heads, uint32_t num_k_heads, uint32_t head_k_dim, uint32_t head_v_dim, uint32_t suffix_len) {
    if (exact_mode()) return false; // reference-order mode: the token-by-token recurrence in the reference's own loop order (k_exact.hip)
    static const uint32_t min_t = [] {
        const char* e = lab_env("UZU_DN_CHUNK_MIN_T");
        return e ? (uint32_t)atoi(e) : 16u; // a prompt of 12 tokens is as fast token by token, one of 63 12 % slower (0.8B model: 2.16 against 1.90 ms)
    }();
    return head_k_dim == DKC && num_k_heads && num_v_heads % num_k_heads == 0 && head_v_dim % 16 == 0 && suffix_len >= min_t;
}

// prep != null: DeltaNetPrefillPrep fused into the chunk preparation (q_norm / k_norm are then OUTPUTS of this call; beta / decay are not materialised)
struct FusedPrep {
    const float *a_log, *dt_bias;
    const uint16_t* conv_rows; // non-null: the conv'd q | k | v channels, [suffix_len][conv_dim] (out-of-place conv)
    float* conv_state;
};
static uzu_status prefill_chunked(hipStream_t s, float* q_norm, float* k_norm, const float* beta, const float* decay, const uint16_t* in_proj, float* state, uint16_t* out,
                                  float* workspace, uint32_t num_v_heads, uint32_t num_k_heads, uint32_t head_v_dim, uint32_t key_dim, uint32_t value_dim, uint32_t suffix_len,
                                  const FusedPrep* prep) {
    const uint32_t n_chunks = (suffix_len + CC - 1) / CC;
    const uint16_t* v_rows = prep && prep->conv_rows ? prep->conv_rows : in_proj; // where the scans read the conv'd v channels
    const uint32_t v_stride = prep && prep->conv_rows ? 2 * key_dim + value_dim : 0u;
    float* const u_ws = workspace + (size_t)n_chunks * num_v_heads * WS_FLOATS; // U
    if (prep)
        UZU_PROPAGATE(launch_check([&] {
            hipLaunchKernelGGL(dn_chunk_prep_kernel<true>, dim3(n_chunks, num_v_heads), dim3(256), 0, s, (const float*)nullptr, (const float*)nullptr, (const float*)nullptr,
                               (const float*)nullptr, workspace, u_ws, num_v_heads, num_k_heads, head_v_dim, key_dim, suffix_len, in_proj, prep->a_log, prep->dt_bias, q_norm, k_norm, value_dim,
                               prep->conv_rows, prep->conv_state);
        }, "delta_net_chunk_prep_fused"));
    else
        UZU_PROPAGATE(launch_check([&] {
            hipLaunchKernelGGL(dn_chunk_prep_kernel<false>, dim3(n_chunks, num_v_heads), dim3(256), 0, s, (const float*)q_norm, (const float*)k_norm, beta, decay, workspace, u_ws,
                               num_v_heads, num_k_heads, head_v_dim, key_dim, suffix_len, in_proj, (const float*)nullptr, (const float*)nullptr, (float*)nullptr,
                               (float*)nullptr, value_dim, (const uint16_t*)nullptr, (float*)nullptr);
        }, "delta_net_chunk_prep"));
    ScanSplit sp{};
    sp.mid_chunk = value_dim == num_v_heads * head_v_dim ? split_mid_chunk(n_chunks, head_v_dim) : 0u;
    static LdsLimit fix_lds;
    if (sp.mid_chunk && !raise_lds_limit(fix_lds, (const void*)dn_chunk_fixup_kernel, kFixLdsBytes)) sp.mid_chunk = 0; // (68 KB of LDS per workgroup)
    if (!sp.mid_chunk)
        return launch_check([&] {
            hipLaunchKernelGGL(dn_chunk_scan_kernel<false>, dim3(head_v_dim / 16, num_v_heads), dim3(256), 0, s, q_norm, k_norm, v_rows, (const float*)workspace, (const float*)u_ws,
                               (const float*)state, state, out, num_v_heads, num_k_heads, head_v_dim, key_dim, value_dim, suffix_len, sp, v_stride);
        }, "delta_net_chunk_scan");
    { // the split's pieces live behind U (delta_net_chunk_workspace_bytes)
        float* w = u_ws + (size_t)n_chunks * CC * value_dim;
        sp.mid_state = w, w += (size_t)value_dim * DKC;
        sp.z_end = w, w += (size_t)value_dim * DKC;
        sp.h_end = w, w += (size_t)num_v_heads * DKC * DKC;
        sp.o32 = w, w += (size_t)suffix_len * value_dim;
        sp.u = w, w += (size_t)suffix_len * num_v_heads * DKC;
        sp.off = (uint32_t*)w;
    }
    UZU_PROPAGATE(launch_check([&] {
        hipLaunchKernelGGL(dn_chunk_scan_kernel<true>, dim3(2 * (head_v_dim / 16), num_v_heads), dim3(512), 0, s, q_norm, k_norm, v_rows, (const float*)workspace, (const float*)u_ws,
                           (const float*)state, state, out, num_v_heads, num_k_heads, head_v_dim, key_dim, value_dim, suffix_len, sp, v_stride);
    }, "delta_net_chunk_scan_dual"));
    const uint32_t t_mid = sp.mid_chunk * CC, t2 = suffix_len - t_mid;
    return launch_check([&] {
        hipLaunchKernelGGL(dn_chunk_fixup_kernel, dim3((t2 + FIX_TOK - 1) / FIX_TOK + DKC / 16, num_v_heads), dim3(256), kFixLdsBytes, s, sp, state, out,
                           num_v_heads, head_v_dim, value_dim, suffix_len, (const float*)q_norm, (const float*)k_norm, v_rows, (const float*)workspace, num_k_heads, key_dim, v_stride);
    }, "delta_net_chunk_fixup");
}

uzu_status delta_net_prefill_chunked(hipStream_t s, const float* q_norm, const float* k_norm, const float* beta, const float* decay, const uint16_t* in_proj,
                                     float* state, uint16_t* out, float* workspace, uint32_t num_v_heads, uint32_t num_k_heads, uint32_t head_v_dim,
                                     uint32_t key_dim, uint32_t value_dim, uint32_t suffix_len) {
    return prefill_chunked(s, (float*)q_norm, (float*)k_norm, beta, decay, in_proj, state, out, workspace, num_v_heads, num_k_heads, head_v_dim, key_dim, value_dim, suffix_len, nullptr);
}
// UZU_HIP_TUNE=prep_fused=0: DeltaNetPrefillPrep as its own launch in front (tests/test_gpu_prefill_switches.py holds the fused kernel to it, bit for bit)
bool delta_net_prefill_prep_fused_enabled() {
    const char* e = tune_env("prep_fused");
    return !e || atoi(e) != 0;
}
uzu_status delta_net_prefill_chunked_fused(hipStream_t s, const uint16_t* in_proj, const float* a_log, const float* dt_bias, float* q_norm_out, float* k_norm_out, float* state,
                                           uint16_t* out, float* workspace, uint32_t num_v_heads, uint32_t num_k_heads, uint32_t head_v_dim, uint32_t key_dim, uint32_t value_dim,
                                           uint32_t suffix_len, const uint16_t* conv_rows, float* conv_state) {
    const FusedPrep prep{a_log, dt_bias, conv_rows, conv_rows ? conv_state : nullptr};
    return prefill_chunked(s, q_norm_out, k_norm_out, nullptr, nullptr, in_proj, state, out, workspace, num_v_heads, num_k_heads, head_v_dim, key_dim, value_dim, suffix_len, &prep);
}

} // namespace k
} // namespace uzu
