// k_deltanet_tree.hip -- Gated DeltaNet over a speculated token TREE (BU = crates/backend-uzu/src).
//
// Reference: ConvTreeScan (BU/backends/cpu/kernel/gdn/tree_verify/conv_scan.rs), DeltaNetPrefillPrep in its tree instantiation
// (gdn/prefill_prep.rs with QKT = T, write_log_decay, write_compact_v: encodable_block/mixer/delta_net.rs:257-265), the
// DeltaNetTreeVerify composite (prefix -> Gram -> solve -> out: backends/metal/kernel/gdn/tree_verify.rs:92-187 over
// cpu/kernel/gdn/tree_verify/{prefix,tree_gram,tree_update_solve,out}.rs) and StateAdvance (tree_verify/state_advance.rs).
//
// Shape of the problem on MI355X: a verify pass carries n <= 32 tree nodes (the reference's stream speculates <= 16), a DeltaNet layer
// has Hv x Dv = 2048 independent output columns, and the only sizeable operand is the f32 state (64 KB per head, streamed ONCE for all
// nodes).  The whole chunked solve of one (head, 16-column tile) is ~n^2 dot products of 128 -- nowhere near worth matrix cores -- so it
// runs as ONE launch of Hv * Dv / 16 workgroups (128 for Qwen3.5) that each stage q / k / their state tile in LDS and walk the
// reference's loops with one thread per output element, sequentially in the reference's order.  That makes the results BIT-IDENTICAL to
// the CPU kernels (no second reference-order variant is needed) at a cost of a few microseconds of dependent latency per launch; three
// launches per layer (prep, solve, norm-gate) against the reference's six.  StateAdvance is the exception: 2048 state rows x <= 16
// sequential delta-rule steps in reference order would be one thread per row (~100 us); the production form gives a row to a half-wave
// (tolerance-class like the decode update), the reference-order form exists for uzu_hip_set_exact(1).
#include "device_utils.h"
#include "silu_near.h"
#include "tree_pass.h"

namespace uzu {
namespace k {

namespace {
constexpr uint32_t kBlock = 16; // token block of the packed-A / inverse tiles (tree_gram.rs:7)

// ------------------------------------------------------------------------------------------------ conv tree scan + tree prep
// grid (slabs, n), 128 threads = one slab of 128 channels of one node.  Slabs [0, Hk): q heads, [Hk, 2Hk): k heads, [2Hk, 2Hk + Hv): value
// heads, slab 2Hk + Hv: the node's per-head scalars (beta, log decay).  head_k_dim == head_v_dim == 128 (delta_net.rs:176-187).
// do_conv: ConvTreeScan on the slab's channels (history walked through `parents`, taps newest first, SiLU); otherwise the rows are read as
// already convolved.  do_prep: l2-normalised q / k ROUNDED to bf16, compact v, beta, log decay.  out_proj (optional, do_conv): the full
// [n, total_proj_dim] rows ConvTreeScan writes (the non-conv channels pass through).
__global__ void __launch_bounds__(128) dn_tree_prep_kernel(const uint16_t* __restrict__ in_proj, const float* __restrict__ conv_w, const float* __restrict__ conv_b,
                                                           const float* __restrict__ base_state, const int32_t* __restrict__ parents, uint16_t* __restrict__ out_proj,
                                                           float* __restrict__ suffix_state, const float* __restrict__ a_log, const float* __restrict__ dt_bias,
                                                           uint16_t* __restrict__ q_out, uint16_t* __restrict__ k_out, uint16_t* __restrict__ v_out, float* __restrict__ beta_out,
                                                           float* __restrict__ log_decay_out, uint32_t n, uint32_t ks, uint32_t Hk, uint32_t Hv, uint32_t do_conv, uint32_t do_prep) {
    constexpr uint32_t D = 128;
    const uint32_t key_dim = Hk * D, value_dim = Hv * D, conv_dim = 2 * key_dim + value_dim, total = conv_dim + value_dim + 2 * Hv;
    const uint32_t slab = blockIdx.x, node = blockIdx.y, c = threadIdx.x, state_stride = ks - 1;
    __shared__ float s_x[D];
    __shared__ float s_inv;
    if (slab == 2 * Hk + Hv) { // per-head scalars + the pass-through channels of ConvTreeScan's output rows
        if (do_conv && out_proj)
            for (uint32_t ch = conv_dim + c; ch < total; ch += D) out_proj[(size_t)node * total + ch] = in_proj[(size_t)node * total + ch];
        if (do_prep && c < Hv) {
            const uint32_t hv = c;
            const float beta_raw = bf16_to_f32(in_proj[(size_t)node * total + conv_dim + value_dim + hv]);
            const float beta = 1.0f / (1.0f + expf_glibc(-beta_raw));
            const float a_raw = bf16_to_f32(in_proj[(size_t)node * total + conv_dim + value_dim + Hv + hv]);
            const float sp_in = a_raw + dt_bias[hv];
            const float sp = sp_in > 20.0f ? sp_in : logf_glibc(1.0f + expf_glibc(sp_in));
            beta_out[(size_t)node * Hv + hv] = beta;
            log_decay_out[(size_t)node * Hv + hv] = -expf_glibc(a_log[hv]) * sp;
        }
        return;
    }
    const uint32_t ch = slab * D + c; // q heads, k heads and value heads are consecutive 128-channel slabs of the conv block
    float xb; // the channel's value as the activation type holds it
    if (do_conv) {
        float acc = conv_b ? conv_b[ch] : 0.0f;
        int32_t source_row = (int32_t)node;
        for (uint32_t h = 0; h < ks; ++h) { // conv_scan.rs:43-65
            float sample;
            if (source_row >= 0) sample = bf16_to_f32(in_proj[(size_t)source_row * total + ch]);
            else sample = base_state[(size_t)ch * state_stride + (state_stride - (uint32_t)(-source_row))];
            acc += sample * conv_w[(size_t)ch * ks + (ks - 1 - h)];
            if (h < state_stride) suffix_state[((size_t)node * conv_dim + ch) * state_stride + (state_stride - 1 - h)] = sample;
            source_row = source_row >= 0 ? parents[source_row] : source_row - 1;
        }
        const uint16_t bits = f32_to_bf16(silu_f32(acc));
        if (out_proj) out_proj[(size_t)node * total + ch] = bits;
        xb = bf16_to_f32(bits);
    } else {
        xb = bf16_to_f32(in_proj[(size_t)node * total + ch]);
    }
    if (!do_prep) return;
    if (slab >= 2 * Hk) { // compact v: the row's value section as it is (prefill_prep.rs:45-52)
        v_out[(size_t)node * value_dim + (slab - 2 * Hk) * D + c] = f32_to_bf16(xb);
        return;
    }
    s_x[c] = xb;
    __syncthreads();
    if (c == 0) { // the reference's sum: sequential from 0 (prefill_prep.rs:57-62, 72-77)
        float sq = 0.0f;
        for (uint32_t j = 0; j < D; ++j) sq += s_x[j] * s_x[j];
        s_inv = 1.0f / sqrtf(sq + 1e-6f);
    }
    __syncthreads();
    const float inv = s_inv;
    if (slab < Hk) {
        const float q_scale = 1.0f / sqrtf((float)D);
        q_out[(size_t)node * key_dim + slab * D + c] = f32_to_bf16(xb * inv * q_scale);
    } else {
        k_out[(size_t)node * key_dim + (slab - Hk) * D + c] = f32_to_bf16(xb * inv);
    }
}

// ------------------------------------------------------------------------------------------------ prefix + Gram + solve + out
// One workgroup = (value head hv, 16 value columns c0 .. c0 + 15), 256 threads, all n nodes.  Every output element is computed by one
// thread walking the reference's loop in the reference's order (see the file header); LDS rows are padded to 132 floats (threads of a
// wave read the same four elements of different rows, 16 bytes at a time).
constexpr uint32_t kPad = 132;
struct alignas(16) TreeSolveLds {
    float q[kDnTreeMaxNodes][kPad];
    float k[kDnTreeMaxNodes][kPad];
    float h0[16][kPad];
    float a[kDnTreeMaxNodes][kDnTreeMaxNodes + 1];   // A[row][col] (strict ancestors), tree_gram.rs:63-96
    float qkd[kDnTreeMaxNodes][kDnTreeMaxNodes + 1]; // tree_gram.rs:44-60
    float a_inv[kDnTreeMaxNodes / kBlock][kBlock][kBlock + 1];
    float kh0[kDnTreeMaxNodes][17], qh0[kDnTreeMaxNodes][17], u[kDnTreeMaxNodes][17];
    float acc[kBlock][17];
    float prefix[kDnTreeMaxNodes], beta[kDnTreeMaxNodes], log_decay[kDnTreeMaxNodes];
    uint32_t t_start[kDnTreeMaxNodes], t_end[kDnTreeMaxNodes];
};
__global__ void __launch_bounds__(256) dn_tree_solve_kernel(const uint16_t* __restrict__ q_in, const uint16_t* __restrict__ k_in, const uint16_t* __restrict__ v_in,
                                                            const uint32_t* __restrict__ trie, const float* __restrict__ log_decay, const float* __restrict__ beta_in,
                                                            const float* __restrict__ h0, uint16_t* __restrict__ o, float scale, uint32_t n, uint32_t Hk, uint32_t Hv) {
    constexpr uint32_t D = 128;
    __shared__ TreeSolveLds L;
    const uint32_t tid = threadIdx.x;
    const uint32_t tiles = D / 16, hv = blockIdx.x / tiles, c0 = (blockIdx.x % tiles) * 16, hk = hv / (Hv / Hk);
    const uint32_t key_dim = Hk * D, value_dim = Hv * D;
    // every global operand is requested up front (round 4: the phases below used to start with a dependent global load each -- log decays inside
    // the prefix loop, v inside the solve -- one exposed L2 / HBM round trip per phase of a 20 us kernel)
    if (tid < n) {
        L.t_start[tid] = trie[3 * tid], L.t_end[tid] = trie[3 * tid + 1];
        L.beta[tid] = beta_in[(size_t)tid * Hv + hv];
        L.log_decay[tid] = log_decay[(size_t)tid * Hv + hv];
    }
    static_assert(kDnTreeMaxNodes / kBlock == 2, "v_pre is selected by hand below");
    float v_pre[kDnTreeMaxNodes / kBlock]; // v of (token blk * kBlock + tid / 16, value column tid % 16), one per block of the solve
#pragma unroll
    for (uint32_t blk = 0; blk < kDnTreeMaxNodes / kBlock; ++blk) {
        const uint32_t token = min(blk * kBlock + tid / 16, n - 1); // clamped: never consumed past n
        v_pre[blk] = bf16_to_f32(v_in[(size_t)token * value_dim + hv * D + c0 + tid % 16]);
    }
    if (((uintptr_t)q_in & 15) == 0 && ((uintptr_t)k_in & 15) == 0 && ((uintptr_t)h0 & 15) == 0) {
        // 16 bytes a lane and every load in front of the first store: element by element, q and k were seven trips to memory one behind the other at 13 nodes (17.4 us, now 13.4, of which ~2 are launch and the rest the chains below)
        static_assert(kDnTreeMaxNodes * D / 8 == 512, "two pieces of 8 q / k elements a thread");
        const uint32_t c = tid % 16 * 8;
        u32x4_v qv[2], kv[2];
        f32x4_v hv4[2];
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i) {
            const size_t at = (size_t)min(tid / 16 + 16 * i, n - 1) * key_dim + hk * D + c;
            qv[i] = *(const u32x4_v*)(q_in + at), kv[i] = *(const u32x4_v*)(k_in + at);
            hv4[i] = *(const f32x4_v*)(h0 + ((size_t)hv * D + c0) * D + (tid + 256 * i) * 4); // 16 consecutive state rows: 8 KB contiguous
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i) {
            const uint32_t row = tid / 16 + 16 * i;
            *(f32x4_v*)&L.h0[(tid + 256 * i) / 32][(tid + 256 * i) % 32 * 4] = hv4[i];
            if (row >= n) continue;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                *(f32x4_v*)&L.q[row][c + 4 * h] = f32x4_v{bits_to_f32(qv[i][2 * h] << 16), bits_to_f32(qv[i][2 * h] & 0xFFFF0000u), bits_to_f32(qv[i][2 * h + 1] << 16), bits_to_f32(qv[i][2 * h + 1] & 0xFFFF0000u)};
                *(f32x4_v*)&L.k[row][c + 4 * h] = f32x4_v{bits_to_f32(kv[i][2 * h] << 16), bits_to_f32(kv[i][2 * h] & 0xFFFF0000u), bits_to_f32(kv[i][2 * h + 1] << 16), bits_to_f32(kv[i][2 * h + 1] & 0xFFFF0000u)};
            }
        }
    } else {
        for (uint32_t idx = tid; idx < n * D; idx += 256) {
            const uint32_t row = idx / D, d = idx % D;
            L.q[row][d] = bf16_to_f32(q_in[(size_t)row * key_dim + hk * D + d]);
            L.k[row][d] = bf16_to_f32(k_in[(size_t)row * key_dim + hk * D + d]);
        }
        for (uint32_t idx = tid; idx < 16 * D; idx += 256) L.h0[idx / D][idx % D] = h0[((size_t)hv * D + c0) * D + idx];
    }
    __syncthreads();
    if (tid < n) { // prefix.rs:20-36: log decays of the ancestors-or-self, in column order
        float sum = 0.0f;
        for (uint32_t col = 0; col < n; ++col)
            if (tid >= L.t_start[col] && tid <= L.t_end[col]) sum += L.log_decay[col];
        L.prefix[tid] = sum;
    }
    __syncthreads();
    for (uint32_t idx = tid; idx < n * n; idx += 256) { // tree_gram.rs:44-96
        const uint32_t row = idx / n, col = idx % n;
        float qkd = 0.0f, a = 0.0f;
        if (row >= L.t_start[col] && row <= L.t_end[col]) {
            // (both sums in one walk, 16 bytes a read: two chains of additions side by side, a quarter of the LDS instructions)
            float qk = 0.0f, kk = 0.0f;
#pragma unroll 4
            for (uint32_t d = 0; d < D; d += 4) {
                const f32x4_v a = *(const f32x4_v*)&L.q[row][d], b = *(const f32x4_v*)&L.k[col][d], c = *(const f32x4_v*)&L.k[row][d];
#pragma unroll
                for (int t = 0; t < 4; ++t) qk += a[t] * b[t], kk += c[t] * b[t];
            }
            const float e = expf_glibc(L.prefix[row] - L.prefix[col]);
            qkd = e * scale * qk;
            if (row != col) a = L.beta[row] * e * kk;
        }
        L.qkd[row][col] = qkd, L.a[row][col] = a;
    }
    for (uint32_t idx = tid; idx < n * 16; idx += 256) { // tree_gram.rs:139-158 (kh0) and the q . h0 term of out.rs:62-73
        const uint32_t token = idx / 16, j = idx % 16;
        float sk = 0.0f, sq = 0.0f;
#pragma unroll 4
        for (uint32_t d = 0; d < D; d += 4) {
            const f32x4_v h = *(const f32x4_v*)&L.h0[j][d], a = *(const f32x4_v*)&L.k[token][d], b = *(const f32x4_v*)&L.q[token][d];
#pragma unroll
            for (int t = 0; t < 4; ++t) sk += a[t] * h[t], sq += b[t] * h[t];
        }
        L.kh0[token][j] = sk, L.qh0[token][j] = sq;
    }
    __syncthreads();
    const uint32_t nb = (n + kBlock - 1) / kBlock;
    if (tid < nb * kBlock) { // tree_gram.rs:98-128: (I + A_diag)^-1 by forward substitution; a thread owns one column of one block
        const uint32_t blk = tid / kBlock, col = tid % kBlock, bs = min(kBlock, n - blk * kBlock);
        float inv[kBlock]; // the thread's column stays in registers (the LDS copy made every row wait for the previous row's store)
#pragma unroll
        for (uint32_t row = 0; row < kBlock; ++row) inv[row] = row == col ? 1.0f : 0.0f;
#pragma unroll
        for (uint32_t row = 1; row < kBlock; ++row) {
            if (row > col && row < bs) {
                float sum = 0.0f;
#pragma unroll
                for (uint32_t prev = 0; prev < row; ++prev)
                    if (prev >= col) sum += L.a[blk * kBlock + row][blk * kBlock + prev] * inv[prev];
                inv[row] = -sum;
            }
        }
#pragma unroll
        for (uint32_t row = 0; row < kBlock; ++row) L.a_inv[blk][row][col] = inv[row];
    }
    __syncthreads();
    const uint32_t lt = tid / 16, j = tid % 16; // (token of the block, value column)
    for (uint32_t blk = 0; blk < nb; ++blk) { // tree_update_solve.rs:58-127
        const uint32_t token = blk * kBlock + lt;
        if (token < n) {
            const float v_val = blk == 0 ? v_pre[0] : v_pre[1]; // (kDnTreeMaxNodes / kBlock == 2 blocks; no dynamic register index)
            float acc = L.beta[token] * (v_val - expf_glibc(L.prefix[token]) * L.kh0[token][j]);
            for (uint32_t prev = 0; prev < blk * kBlock; ++prev) acc -= L.a[token][prev] * L.u[prev][j];
            L.acc[lt][j] = acc;
        }
        __syncthreads();
        if (token < n) {
            float sum = 0.0f;
            for (uint32_t lp = 0; lp < kBlock && blk * kBlock + lp < n; ++lp) sum += L.a_inv[blk][lt][lp] * L.acc[lp][j];
            L.u[token][j] = sum;
        }
        __syncthreads();
    }
    for (uint32_t idx = tid; idx < n * 16; idx += 256) { // out.rs:55-84
        const uint32_t row = idx / 16, jj = idx % 16;
        float acc = 0.0f;
        acc += expf_glibc(L.prefix[row]) * scale * L.qh0[row][jj];
        for (uint32_t col = 0; col < n; ++col) acc += L.qkd[row][col] * L.u[col][jj];
        o[(size_t)row * value_dim + hv * D + c0 + jj] = f32_to_bf16(acc);
    }
}

// ------------------------------------------------------------------------------------------------ the pass in one launch
// Conv scan, preparation, prefix, Gram, solve and out of a verify pass: dn_tree_prep_kernel and dn_tree_solve_kernel in one launch, every value by the same operations in the
// same order, so bit-identical to the two (and to the CPU kernels).  What they cost was trips to memory and idle lanes, not work: the preparation walked the parents by
// dependent loads, its rows went out and came back, and 256 threads took the 128-long sums of one after the other (20.5 us a layer at 13 nodes, now 11.4).
// One workgroup = (value head hv, 16 value columns), 1024 threads, all n nodes.  It convolves its head's q and k channels for itself, eight workgroups of a head the same:
// 13 x 256 channels are 2.8 us of a compute unit, the launch and the trips that they replace 6.8.  Tile t of a head files the nodes t, t + 8, ... for the acceptance that follows.
constexpr uint32_t kTreeStepMaxKernel = 4; // taps: the history of a channel in registers, a node's source rows in a byte each
struct alignas(16) TreeStepLds {
    float q[kDnTreeMaxNodes][kPad];
    float k[kDnTreeMaxNodes][kPad];
    float h0[16][kPad];
    uint16_t x[kDnTreeMaxNodes][272]; // the rows' q, k and the tile's v channels in front of the convolution
    float a[kDnTreeMaxNodes][kDnTreeMaxNodes + 4]; // (rows of 16 bytes' multiples)
    float qkd[kDnTreeMaxNodes][kDnTreeMaxNodes + 4];
    float a_inv[kDnTreeMaxNodes / kBlock][kBlock][kBlock + 4];
    float v[kDnTreeMaxNodes][17], kh0[kDnTreeMaxNodes][17], qh0[kDnTreeMaxNodes][17], u[kDnTreeMaxNodes][17];
    float acc[kBlock][17];
    float prefix[kDnTreeMaxNodes], e_prefix[kDnTreeMaxNodes], beta[kDnTreeMaxNodes], inv[2][kDnTreeMaxNodes];
    uint64_t exp_tab[32];
    uint32_t rows[kDnTreeMaxNodes]; // a node's source rows, newest tap first, a signed byte each: a node, or -1, -2, -3 into the sequence's history
    uint32_t t_start[kDnTreeMaxNodes], t_end[kDnTreeMaxNodes];
};
template <uint32_t KS>
__global__ void __launch_bounds__(1024) dn_tree_step_kernel(const uint16_t* __restrict__ in_proj, const float* __restrict__ conv_w, const float* __restrict__ conv_b,
                                                            const float* __restrict__ base_state, const int32_t* __restrict__ parents, const uint32_t* __restrict__ trie,
                                                            const float* __restrict__ a_log, const float* __restrict__ dt_bias, const float* __restrict__ h0,
                                                            float* __restrict__ suffix_state, uint16_t* __restrict__ k_out, uint16_t* __restrict__ v_out,
                                                            float* __restrict__ beta_out, float* __restrict__ log_decay_out, uint16_t* __restrict__ o, uint32_t n, uint32_t Hk,
                                                            uint32_t Hv) {
    constexpr uint32_t D = 128, T = 1024, tiles = D / 16, history = KS - 1, kGroups = 3;
    __shared__ TreeStepLds L;
    const uint32_t tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, hv = blockIdx.x / tiles, t = blockIdx.x % tiles, c0 = t * 16, hk = hv / (Hv / Hk);
    const uint32_t key_dim = Hk * D, value_dim = Hv * D, conv_dim = 2 * key_dim + value_dim, total = conv_dim + value_dim + 2 * Hv;
    const bool files_k = hv % (Hv / Hk) == 0; // (value heads that share a key head: the first of them files it)
    // ---- every operand is requested before the first is used
    // rows: 16 bytes a thread, 16 pieces of q and 16 of k a node, and two of v
    const uint32_t x_node = min(tid / 32, n - 1), x_piece = tid % 32, xv_node = min(tid / 2, n - 1);
    const u32x4_v x = *(const u32x4_v*)(in_proj + (size_t)x_node * total + (x_piece < 16 ? 0 : key_dim) + hk * D + x_piece % 16 * 8);
    u32x4_v xv = {0u, 0u, 0u, 0u};
    if (wave == 0) xv = *(const u32x4_v*)(in_proj + (size_t)xv_node * total + 2 * key_dim + hv * D + c0 + tid % 2 * 8);
    f32x4_v state = {0.f, 0.f, 0.f, 0.f};
    if (wave < 8) state = *(const f32x4_v*)(h0 + ((size_t)hv * D + c0) * D + tid * 4);
    // the convolution's roles: waves 0 .. 11 a q or k channel a thread, three groups of nodes; 12 .. 14 a value channel, twelve nodes at a time; the last one the nodes' scalars
    const uint32_t c = tid % 256, channel = wave < 12 ? (c < D ? 0 : key_dim) + hk * D + c % D : 2 * key_dim + hv * D + c0 + tid % 16;
    float w[KS], past[history];
#pragma unroll
    for (uint32_t i = 0; i < KS; ++i) w[i] = conv_w[(size_t)channel * KS + i];
#pragma unroll
    for (uint32_t i = 0; i < history; ++i) past[i] = base_state[(size_t)channel * history + i];
    const float bias = conv_b ? conv_b[channel] : 0.0f;
    float beta_raw = 0.f, a_raw = 0.f, bias_dt = 0.f, log_a = 0.f;
    uint32_t start = 1, end = 0;
    if (wave == 15 && lane < n) {
        beta_raw = bf16_to_f32(in_proj[(size_t)lane * total + conv_dim + value_dim + hv]);
        a_raw = bf16_to_f32(in_proj[(size_t)lane * total + conv_dim + value_dim + Hv + hv]);
        bias_dt = dt_bias[hv], log_a = a_log[hv];
        start = trie[3 * lane], end = trie[3 * lane + 1];
        L.t_start[lane] = start, L.t_end[lane] = end;
    }
    if (wave == 14 && lane < n) { // conv_scan.rs:43-65: the node, its ancestors, then the history backwards
        int32_t row = (int32_t)lane;
        uint32_t packed = 0;
#pragma unroll
        for (uint32_t h = 0; h < KS; ++h) {
            packed |= ((uint32_t)row & 255u) << (8 * h);
            if (h + 1 < KS) row = row >= 0 ? parents[row] : row - 1;
        }
        L.rows[lane] = packed;
    }
    if (tid < 32) L.exp_tab[tid] = kExp2fTab[tid];
    for (uint32_t i = tid; i < kDnTreeMaxNodes * (kDnTreeMaxNodes + 4); i += T) (&L.a[0][0])[i] = 0.0f, (&L.qkd[0][0])[i] = 0.0f;
    if (tid / 32 < n) *(u32x4_v*)&L.x[tid / 32][x_piece * 8] = x;
    if (tid < 2 * n) *(u32x4_v*)&L.x[tid / 2][256 + tid % 2 * 8] = xv;
    if (wave < 8) *(f32x4_v*)&L.h0[tid / 32][tid % 32 * 4] = state;
    __syncthreads();
    auto convolve = [&](uint32_t node, uint32_t packed, uint32_t at, bool files) { // taps newest first
        float acc = bias;
#pragma unroll
        for (uint32_t h = 0; h < KS; ++h) {
            const int32_t row = (int32_t)(packed << (24 - 8 * h)) >> 24;
            float sample = bf16_to_f32(L.x[max(row, 0)][at]);
#pragma unroll
            for (uint32_t i = 0; i < history; ++i) sample = row == (int32_t)i - (int32_t)history ? past[i] : sample;
            acc += sample * w[KS - 1 - h];
            if (files && h < history) suffix_state[((size_t)node * conv_dim + channel) * history + (history - 1 - h)] = sample;
        }
        return silu_bf16(acc, L.exp_tab);
    };
    if (wave < 4 * kGroups) {
        for (uint32_t node = wave / 4; node < n; node += kGroups) {
            const float xb = bf16_to_f32(convolve(node, __builtin_amdgcn_readfirstlane(L.rows[node]), c, files_k && node % tiles == t));
            if (c < D) L.q[node][c] = xb;
            else L.k[node][c - D] = xb;
        }
    } else if (wave < 15) {
        for (uint32_t node = (tid - 256 * kGroups) / 16; node < n; node += 12) {
            const uint16_t bits = convolve(node, L.rows[node], 256 + tid % 16, true);
            L.v[node][tid % 16] = bf16_to_f32(bits);
            v_out[(size_t)node * value_dim + hv * D + c0 + tid % 16] = bits;
        }
    } else {
        const float beta = 1.0f / (1.0f + expf_glibc_tab(-beta_raw, L.exp_tab));
        const float sp_in = a_raw + bias_dt;
        const float sp = sp_in > 20.0f ? sp_in : logf_glibc(1.0f + expf_glibc_tab(sp_in, L.exp_tab));
        const float decay = -expf_glibc_tab(log_a, L.exp_tab) * sp;
        float sum = 0.0f; // prefix.rs:20-36: log decays of the ancestors-or-self, in column order
        for (uint32_t col = 0; col < n; ++col) {
            const uint32_t first = __builtin_amdgcn_readlane(start, col), last = __builtin_amdgcn_readlane(end, col);
            const float with = sum + bits_to_f32(__builtin_amdgcn_readlane(f32_to_bits(decay), col));
            sum = lane >= first && lane <= last ? with : sum;
        }
        if (lane < n) {
            L.beta[lane] = beta, L.prefix[lane] = sum, L.e_prefix[lane] = expf_glibc_tab(sum, L.exp_tab);
            if (t == 0) beta_out[(size_t)lane * Hv + hv] = beta, log_decay_out[(size_t)lane * Hv + hv] = decay;
        }
    }
    __syncthreads();
    // a sum of 128 products in their order: the reads of the next 16 are on their way while the adders work (waited for two by two: 4400 cycles a round of sums, now 3200)
    auto dot = [&](const float* left, const float* right) {
        f32x4_v l[2][4], r[2][4];
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) l[0][i] = *(const f32x4_v*)(left + 4 * i), r[0][i] = *(const f32x4_v*)(right + 4 * i);
#pragma unroll
        for (uint32_t d = 0; d < D; d += 16) {
            const int now = d / 16 % 2;
            if (d + 16 < D) {
#pragma unroll
                for (int i = 0; i < 4; ++i) l[now ^ 1][i] = *(const f32x4_v*)(left + d + 16 + 4 * i), r[now ^ 1][i] = *(const f32x4_v*)(right + d + 16 + 4 * i);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) sum += l[now][i][e] * r[now][i][e];
            asm volatile("" : "+v"(sum)); // (here, not behind all the reads)
        }
        return sum;
    };
    if (tid < 2 * n) { // the reference's sums of squares: sequential from 0 (prefill_prep.rs:57-62, 72-77)
        const float* row = tid < n ? L.q[tid] : L.k[tid - n];
        L.inv[tid < n ? 0 : 1][tid < n ? tid : tid - n] = 1.0f / sqrtf(dot(row, row) + 1e-6f);
    }
    __syncthreads();
    for (uint32_t node = tid / 256; node < n; node += T / 256) {
        if (c < D) {
            const float q_scale = 1.0f / sqrtf((float)D);
            L.q[node][c] = bf16_to_f32(f32_to_bf16(L.q[node][c] * L.inv[0][node] * q_scale));
        } else {
            const uint16_t bits = f32_to_bf16(L.k[node][c - D] * L.inv[1][node]);
            L.k[node][c - D] = bf16_to_f32(bits);
            if (files_k && node % tiles == t) k_out[(size_t)node * key_dim + hk * D + c - D] = bits;
        }
    }
    __syncthreads();
    // ---- the 128-long sums, one a thread: q . k and k . k of the pairs row >= col (tree_gram.rs:44-96; an ancestor comes first), k . h0 and q . h0 (tree_gram.rs:139-158,
    // out.rs:62-73)
    const uint32_t pairs = n * (n + 1) / 2;
    for (uint32_t i = tid; i < 2 * pairs + 32 * n; i += T) {
        uint32_t row, col;
        const float *left, *right;
        const bool pair = i < 2 * pairs;
        const uint32_t which = pair ? (i < pairs ? 0u : 1u) : (i - 2 * pairs < 16 * n ? 0u : 1u); // 0: q with k, k with h0; 1: k with k, q with h0
        if (pair) {
            const uint32_t p = which ? i - pairs : i;
            row = (uint32_t)((sqrtf((float)(8 * p + 1)) - 1.0f) * 0.5f);
            if (row * (row + 1) / 2 > p) --row;
            else if ((row + 1) * (row + 2) / 2 <= p) ++row;
            col = p - row * (row + 1) / 2;
            left = which ? L.k[row] : L.q[row], right = L.k[col];
        } else {
            const uint32_t p = i - 2 * pairs - which * 16 * n;
            row = p / 16, col = p % 16;
            left = which ? L.q[row] : L.k[row], right = L.h0[col];
        }
        const float sum = dot(left, right);
        if (!pair) {
            (which ? L.qh0 : L.kh0)[row][col] = sum;
        } else if (row >= L.t_start[col] && row <= L.t_end[col]) {
            const float e = expf_glibc_tab(L.prefix[row] - L.prefix[col], L.exp_tab);
            if (!which) L.qkd[row][col] = e * 1.0f * sum; // (the composite's scale: q carries its own)
            else if (row != col) L.a[row][col] = L.beta[row] * e * sum;
        }
    }
    __syncthreads();
    const uint32_t nb = (n + kBlock - 1) / kBlock;
    const uint32_t lt = (tid & 255) / 16, j = tid % 16; // (token of the block, value column)
    if (wave == 0) { // tree_gram.rs:98-128: (I + A_diag)^-1 by forward substitution; a thread owns one column of one block (rows past the last node: of zeros)
        const uint32_t blk = lane / kBlock % (kDnTreeMaxNodes / kBlock), col = lane % kBlock;
        float inv[kBlock];
        f32x4_v a[2][kBlock / 4]; // a row and the one behind it
        auto read = [&](uint32_t row) {
#pragma unroll
            for (uint32_t i = 0; 4 * i < row; ++i) a[row % 2][i] = *(const f32x4_v*)&L.a[blk * kBlock + row][blk * kBlock + 4 * i];
        };
#pragma unroll
        for (uint32_t row = 0; row < kBlock; ++row) {
            if (row + 1 < kBlock) read(row + 1);
            __builtin_amdgcn_sched_barrier(0);
            float sum = 0.0f;
#pragma unroll
            for (uint32_t prev = 0; prev < row; ++prev) {
                const float with = sum + a[row % 2][prev / 4][prev % 4] * inv[prev];
                sum = prev >= col ? with : sum;
            }
            inv[row] = row > col ? -sum : row == col ? 1.0f : 0.0f;
            asm volatile("" : "+v"(inv[row]));
        }
        if (lane < kDnTreeMaxNodes) {
#pragma unroll
            for (uint32_t row = 0; row < kBlock; ++row) L.a_inv[blk][row][col] = inv[row];
        }
    } else if (tid >= 256 && tid < 512 && lt < n) { // tree_update_solve.rs:58-127, the first block's right-hand side meanwhile
        L.acc[lt][j] = L.beta[lt] * (L.v[lt][j] - L.e_prefix[lt] * L.kh0[lt][j]);
    }
    __syncthreads();
    for (uint32_t blk = 0; blk < nb; ++blk) {
        const uint32_t token = blk * kBlock + lt;
        if (blk) {
            if (tid < 256 && token < n) {
                float acc = L.beta[token] * (L.v[token][j] - L.e_prefix[token] * L.kh0[token][j]);
#pragma unroll
                for (uint32_t prev = 0; prev < kBlock; ++prev) acc -= L.a[token][prev] * L.u[prev][j]; // (kDnTreeMaxNodes / kBlock == 2: one block in front)
                L.acc[lt][j] = acc;
            }
            __syncthreads();
        }
        if (tid < 256 && token < n) {
            float sum = 0.0f;
#pragma unroll
            for (uint32_t lp = 0; lp < kBlock; ++lp) {
                const float with = sum + L.a_inv[blk][lt][lp] * L.acc[lp][j];
                sum = blk * kBlock + lp < n ? with : sum;
            }
            L.u[token][j] = sum;
        }
        __syncthreads();
    }
    static_assert(kDnTreeMaxNodes / kBlock == 2, "the second block has one block in front of it");
    if (tid / 16 < n) { // out.rs:55-84
        const uint32_t row = tid / 16;
        float acc = 0.0f;
        acc += L.e_prefix[row] * 1.0f * L.qh0[row][j];
        for (uint32_t col0 = 0; col0 < n; col0 += 8)
#pragma unroll
            for (uint32_t col = col0; col < col0 + 8; ++col) {
                const float with = acc + L.qkd[row][col] * L.u[col][j];
                acc = col < n ? with : acc;
            }
        o[(size_t)row * value_dim + hv * D + c0 + j] = f32_to_bf16(acc);
    }
}

// ------------------------------------------------------------------------------------------------ state advance
// state_advance.rs:25-58.  Production: a state row (hv, dv) lives in the registers of a half-wave (4 consecutive dk per lane) across the
// accepted path; per accepted node: decay, k . row (butterfly over the 32 lanes), delta, rank-one update.
__device__ __forceinline__ void state_advance(const uint16_t* __restrict__ k_norm, const uint16_t* __restrict__ v, const float* __restrict__ log_decay, const float* __restrict__ beta,
                                              const uint32_t* accepted, float* __restrict__ state, uint32_t accepted_len, uint32_t Hv, uint32_t Hk) {
    constexpr uint32_t D = 128;
    const uint32_t row = blockIdx.x * 8 + threadIdx.x / 32, sub = threadIdx.x % 32; // 8 state rows per workgroup
    const uint32_t hv = row / D, dv = row % D, hk = hv / (Hv / Hk);
    float* srow = state + (size_t)row * D + sub * 4;
    f32x4_v st = *(const f32x4_v*)srow;
    for (uint32_t ai = 0; ai < accepted_len; ++ai) {
        const uint32_t node = accepted[ai];
        const float decay = expf_glibc(log_decay[(size_t)node * Hv + hv]);
        const float b = beta[(size_t)node * Hv + hv];
        const u32x2_v kb = *(const u32x2_v*)(k_norm + (size_t)node * Hk * D + hk * D + sub * 4);
        const float k0 = bits_to_f32(kb.x << 16), k1 = bits_to_f32(kb.x & 0xFFFF0000u), k2 = bits_to_f32(kb.y << 16), k3 = bits_to_f32(kb.y & 0xFFFF0000u);
        st.x *= decay, st.y *= decay, st.z *= decay, st.w *= decay;
        float part = ((st.x * k0 + st.y * k1) + st.z * k2) + st.w * k3;
        part = xadd1(part), part = xadd2(part), part = xadd4(part), part = xadd8(part);
        part += __shfl_xor(part, 16, 64); // the two rows of 16 lanes of this half-wave
        const float v_val = bf16_to_f32(v[(size_t)node * Hv * D + hv * D + dv]);
        const float delta = b * (v_val - part);
        st.x += k0 * delta, st.y += k1 * delta, st.z += k2 * delta, st.w += k3 * delta;
    }
    *(f32x4_v*)srow = st;
}
__global__ void __launch_bounds__(256) dn_state_advance_kernel(const uint16_t* __restrict__ k_norm, const uint16_t* __restrict__ v, const float* __restrict__ log_decay,
                                                               const float* __restrict__ beta, const uint32_t* __restrict__ accepted, float* __restrict__ state,
                                                               uint32_t accepted_len, uint32_t Hv, uint32_t Hk) {
    state_advance(k_norm, v, log_decay, beta, accepted, state, accepted_len, Hv, Hk);
}
// The layers' states in one launch, grid.y = layers: a megabyte of state a layer is less than a launch (18 layers of 16 heads: 66 us in 18 launches, now 13; the indices come as
// arguments, which saves their copy)
__global__ void __launch_bounds__(256) dn_states_advance_kernel(TreeStates t) {
    const TreeState& L = t.layer[blockIdx.y];
    if (blockIdx.x * 8 >= L.Hv * 128) return; // (layers of fewer heads)
    state_advance(L.k, L.v, L.log_decay, L.beta, t.accepted, L.state, t.accepted_len, L.Hv, L.Hk);
}
// reference order: one thread per state row, everything sequential (uzu_hip_set_exact)
__global__ void __launch_bounds__(64) dn_state_advance_exact_kernel(const uint16_t* k_norm, const uint16_t* v, const float* log_decay, const float* beta, const uint32_t* accepted,
                                                                    float* state, uint32_t accepted_len, uint32_t Hv, uint32_t Hk) {
    constexpr uint32_t D = 128;
    const uint32_t row = blockIdx.x * 64 + threadIdx.x;
    if (row >= Hv * D) return;
    const uint32_t hv = row / D, dv = row % D, hk = hv / (Hv / Hk);
    float* srow = state + (size_t)row * D;
    for (uint32_t ai = 0; ai < accepted_len; ++ai) {
        const uint32_t node = accepted[ai];
        const float decay = expf_glibc(log_decay[(size_t)node * Hv + hv]);
        const float b = beta[(size_t)node * Hv + hv];
        const uint16_t* kr = k_norm + (size_t)node * Hk * D + hk * D;
        float kv_mem = 0.0f;
        for (uint32_t d = 0; d < D; ++d) {
            srow[d] *= decay;
            kv_mem += srow[d] * bf16_to_f32(kr[d]);
        }
        const float delta = b * (bf16_to_f32(v[(size_t)node * Hv * D + hv * D + dv]) - kv_mem);
        for (uint32_t d = 0; d < D; ++d) srow[d] += bf16_to_f32(kr[d]) * delta;
    }
}
} // namespace

static uzu_status check_dims(const char* what, uint32_t n, uint32_t Hk, uint32_t Hv, uint32_t Dk, uint32_t Dv) {
    if (Dk != 128 || Dv != 128 || !Hk || !Hv || Hv % Hk) { // delta_net.rs:176-187
        set_error("%s: head_dim and value_head_dim must be 128 and value heads a multiple of key heads (got %u / %u, %u / %u heads)", what, Dk, Dv, Hk, Hv);
        return UZU_ERR_UNSUPPORTED;
    }
    if (n > kDnTreeMaxNodes) {
        set_error("%s: a verify pass carries at most %u tree nodes (got %u)", what, kDnTreeMaxNodes, n);
        return UZU_ERR_UNSUPPORTED;
    }
    return UZU_OK;
}

uzu_status delta_net_tree_prep(hipStream_t s, const uint16_t* in_proj, const float* conv_w, const float* conv_b, const float* base_state, const int32_t* parents,
                               uint16_t* out_proj, float* suffix_state, const float* a_log, const float* dt_bias, uint16_t* q_out, uint16_t* k_out, uint16_t* v_out,
                               float* beta_out, float* log_decay_out, uint32_t n, uint32_t kernel_size, uint32_t Hk, uint32_t Hv, uint32_t Dk, uint32_t Dv, bool do_conv,
                               bool do_prep) {
    if (!n) return UZU_OK;
    UZU_PROPAGATE(check_dims("delta_net_tree_prep", n, Hk, Hv, Dk, Dv));
    if (do_conv && kernel_size < 2) {
        set_error("conv_tree_scan: kernel_size must be >= 2");
        return UZU_ERR_INVALID_ARGUMENT;
    }
    return launch_check([&] {
        hipLaunchKernelGGL(dn_tree_prep_kernel, dim3(2 * Hk + Hv + 1, n), dim3(128), 0, s, in_proj, conv_w, conv_b, base_state, parents, out_proj, suffix_state, a_log, dt_bias,
                           q_out, k_out, v_out, beta_out, log_decay_out, n, kernel_size, Hk, Hv, do_conv ? 1u : 0u, do_prep ? 1u : 0u);
    }, "dn_tree_prep");
}

uzu_status delta_net_tree_verify(hipStream_t s, const uint16_t* q, const uint16_t* k, const uint16_t* v, const uint32_t* trie, const float* log_decay, const float* beta,
                                 const float* h0, uint16_t* out, uint32_t n, uint32_t Hk, uint32_t Hv, uint32_t Dk, uint32_t Dv) {
    if (!n) return UZU_OK;
    UZU_PROPAGATE(check_dims("delta_net_tree_verify", n, Hk, Hv, Dk, Dv));
    return launch_check([&] { hipLaunchKernelGGL(dn_tree_solve_kernel, dim3(Hv * (Dv / 16)), dim3(256), 0, s, q, k, v, trie, log_decay, beta, h0, out, 1.0f, n, Hk, Hv); },
                        "dn_tree_solve");
}

bool delta_net_tree_step_supported(const uint16_t* in_proj, const float* h0, uint32_t n, uint32_t kernel_size, uint32_t Hk, uint32_t Hv, uint32_t Dk, uint32_t Dv) {
    return n && n <= kDnTreeMaxNodes && kernel_size >= 2 && kernel_size <= kTreeStepMaxKernel && Dk == 128 && Dv == 128 && Hk && Hv && Hv % Hk == 0 && Hv % 4 == 0 /* rows of 16 bytes' multiples */ &&
           (((uintptr_t)in_proj | (uintptr_t)h0) & 15) == 0;
}
// A workgroup has a CU to itself (82 KB of LDS), so from 33 heads on they come in rounds of 32 heads, and it depends on the nodes what a round more costs.  Us, the two launches and this one:
// 32 heads, 2 / 13 / 32 nodes 12.2 / 7.9, 18.0 / 10.4, 31.4 / 18.9; 48 heads, 2 / 8 / 16 / 17 / 28 / 32 nodes 12.8 / 14.4, 14.8 / 16.3, 20.7 / 20.8, 25.9 / 22.8, 32.4 / 31.7, 33.2 / 34.9, of 64 heads
// within 0.4 of these; 72 heads, 2 / 10 / 13 / 32 nodes 18.5 / 20.8, 25.3 / 25.5, 29.6 / 27.7, 57.3 / 51.3.
bool delta_net_tree_step_faster(uint32_t n, uint32_t Hv) { return Hv <= 32 || (Hv <= 64 ? n > 16 && n <= 28 : n > 10); }
uzu_status delta_net_tree_step(hipStream_t s, const uint16_t* in_proj, const float* conv_w, const float* conv_b, const float* base_state, const int32_t* parents, const uint32_t* trie,
                               const float* a_log, const float* dt_bias, const float* h0, float* suffix_state, uint16_t* k_out, uint16_t* v_out, float* beta_out, float* log_decay_out,
                               uint16_t* out, uint32_t n, uint32_t kernel_size, uint32_t Hk, uint32_t Hv) {
    return launch_check([&] {
        const auto step = kernel_size == 4 ? dn_tree_step_kernel<4> : kernel_size == 3 ? dn_tree_step_kernel<3> : dn_tree_step_kernel<2>;
        hipLaunchKernelGGL(step, dim3(Hv * 8), dim3(1024), 0, s, in_proj, conv_w, conv_b, base_state, parents, trie, a_log, dt_bias, h0, suffix_state, k_out, v_out, beta_out, log_decay_out, out,
                           n, Hk, Hv);
    }, "dn_tree_step");
}

uzu_status delta_net_state_advance(hipStream_t s, const uint16_t* k_norm, const uint16_t* v, const float* log_decay, const float* beta, const uint32_t* accepted_indices,
                                   float* state, uint32_t accepted_len, uint32_t Hv, uint32_t Hk, uint32_t Dk) {
    if (!accepted_len) return UZU_OK;
    UZU_PROPAGATE(check_dims("state_advance", 0, Hk, Hv, Dk, Dk));
    if (exact_mode())
        return launch_check([&] {
            hipLaunchKernelGGL(dn_state_advance_exact_kernel, dim3((Hv * Dk + 63) / 64), dim3(64), 0, s, k_norm, v, log_decay, beta, accepted_indices, state, accepted_len, Hv, Hk);
        }, "dn_state_advance_exact");
    return launch_check([&] {
        hipLaunchKernelGGL(dn_state_advance_kernel, dim3(Hv * Dk / 8), dim3(256), 0, s, k_norm, v, log_decay, beta, accepted_indices, state, accepted_len, Hv, Hk);
    }, "dn_state_advance");
}

uzu_status delta_net_states_advance(hipStream_t s, const TreeStates& t, uint32_t layers) {
    uint32_t heads = 0;
    for (uint32_t l = 0; l < layers; ++l) {
        UZU_PROPAGATE(check_dims("state_advance", 0, t.layer[l].Hk, t.layer[l].Hv, 128, 128));
        heads = heads > t.layer[l].Hv ? heads : t.layer[l].Hv;
    }
    if (!layers || !t.accepted_len) return UZU_OK;
    return launch_check([&] { hipLaunchKernelGGL(dn_states_advance_kernel, dim3(heads * 16, layers), dim3(256), 0, s, t); }, "dn_states_advance");
}

} // namespace k
} // namespace uzu
