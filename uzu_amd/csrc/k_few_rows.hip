// k_few_rows.hip -- linears and experts of the f32-stream designs for a pass of a few rows (bf16 products; linears of 3 to 32 rows, experts of 2 to 63): register-fed matrix cores.
//
// At these sizes a product is its weights' way from memory: 7712 x 2048 is 32 MB, 6 us of reading, and 8 rows of it 0.25 GFLOP.  A wave per output column on the VALU
// (k_stream32.hip, linear_rows) reads a weight once per four rows and pays a conversion and four multiply-adds for it: 26 us.  Here
//   * a workgroup owns 16 NB output columns, its waves share the contraction in chunks of 64 (wave w takes chunks w, w + W, ..: together they read whole rows), and the
//     waves' f32 sums meet once, in LDS, in pairs;
//   * a chunk is two v_mfma_f32_16x16x32_bf16 per 16 columns and 16 rows: lane (r, g) loads 32 bytes of weight row r at 16 g and the same 16 elements of activation row r
//     (f32, rounded to bf16 in registers, from the L2) -- the contraction's order inside a chunk is free as long as both operands share it, and a weight row's 128 bytes
//     are taken whole;
//   * nothing is staged and the next chunks' loads are in flight while a pair is computed.
// What bounds it: memory for wide outputs, the launch and two or three loads' latency for narrow ones (64 to 128 workgroups cannot draw the whole chip's bandwidth).
// Measured, us per launch, a wave per column -> here: 8 rows of 7712 x 2048 23.4 -> 8.6, of 32768 x 2048 91 -> 27.3 (4.9 TB/s), of 2048 x 4096 13.4 -> 10.6, of 4112 x 1024
// 9.1 -> 5.6; 16 rows of 32768 x 2048 184 -> 32; 17 rows of 2048 x 2048 210 (VALU tile) -> 10.9.  Experts of 8 rows, two each of eight, 2048 wide: first product 72 -> 29,
// second 24 -> 16.2 + 4.5 for the sum over a row's winners.
#include "gemm_convert.h"
#include "stream32_epilogue.h"

namespace uzu {
namespace k {

namespace {
typedef __attribute__((ext_vector_type(4))) float fw_f32x4;
constexpr uint32_t kChunk = 64; // elements of the contraction: 128 bytes of a weight row

template <int NB, int MT, int U> struct FewBatch {
    u32x4_t w[U][NB][2];
    fw_f32x4 x[U][MT][4];
};
// wp / xp: this lane's weight row / activation row, already at 8 * (lane >> 4)
template <int NB, int MT, int U>
__device__ __forceinline__ void few_load(FewBatch<NB, MT, U>& b, const uint16_t* const (&wp)[NB], const float* const (&xp)[MT], uint32_t c, uint32_t step, uint32_t last) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t at = c + u * step, k0 = (at < last ? at : last) * kChunk; // (behind the end: the last chunk again, never multiplied)
#pragma unroll
        for (int j = 0; j < NB; ++j) b.w[u][j][0] = *(const u32x4_t*)(wp[j] + k0), b.w[u][j][1] = *(const u32x4_t*)(wp[j] + k0 + 32);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int t = 0; t < 4; ++t) b.x[u][i][t] = *(const fw_f32x4*)(xp[i] + k0 + 32 * (t >> 1) + 4 * (t & 1));
    }
}
__device__ __forceinline__ u32x4_t few_pack(const fw_f32x4& a, const fw_f32x4& b) { return u32x4_t{pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3]), pack_bf16(b[0], b[1]), pack_bf16(b[2], b[3])}; }
// acc[j][i]: lane (m, g), element t = column 16 j + 4 g + t of row 16 i + m.  The matrix core's sums fall short of the exact ones by a rounding that is always downwards: a chain of
// them through the contraction adds up (8 rows of 2048 x 4096: 1.4e-7 of the result's norm against 64 bits; a wave per column 8.4e-8).  So a chunk's two products are summed from
// zero, one of them negated, and their difference added: what is missing of both goes out.
template <int NB, int MT> __device__ __forceinline__ void few_chunk(fw_f32x4 (&acc)[NB][MT], const u32x4_t (&w)[NB][2], const fw_f32x4 (&x)[MT][4]) {
    const fw_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const bf16x8_t b0 = __builtin_bit_cast(bf16x8_t, few_pack(x[i][0], x[i][1])), b1 = __builtin_bit_cast(bf16x8_t, few_pack(-x[i][2], -x[i][3]));
        fw_f32x4 s0[NB], s1[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) s0[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w[j][0]), b0, zero, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NB; ++j) s1[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w[j][1]), b1, zero, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[j][i] += s0[j] - s1[j];
    }
}
template <int NB, int MT, int U>
__device__ __forceinline__ void few_contract(fw_f32x4 (&acc)[NB][MT], const uint16_t* const (&wp)[NB], const float* const (&xp)[MT], uint32_t chunks, uint32_t wave, uint32_t waves) {
    FewBatch<NB, MT, U> a, b;
    const uint32_t step = U * waves, last = chunks - 1;
    auto run = [&](const FewBatch<NB, MT, U>& t, uint32_t c) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c + u * waves < chunks) few_chunk<NB, MT>(acc, t.w[u], t.x[u]);
    };
    if (wave >= chunks) return;
    uint32_t c = wave;
    few_load<NB, MT, U>(a, wp, xp, c, waves, last);
    for (;;) { // (a batch is loaded only where it is multiplied, and never behind a branch that joins in front of a use: such a join waits for everything in flight)
        if (c + step >= chunks) return run(a, c);
        few_load<NB, MT, U>(b, wp, xp, c + step, waves, last);
        __builtin_amdgcn_sched_barrier(0);
        run(a, c);
        c += step;
        if (c + step >= chunks) return run(b, c);
        few_load<NB, MT, U>(a, wp, xp, c + step, waves, last);
        __builtin_amdgcn_sched_barrier(0);
        run(b, c);
        c += step;
    }
}
// the waves' sums into LDS ([wave][tile][lane][4]); element e of the summed tiles afterwards
template <int T> __device__ __forceinline__ void few_put(float* s_sum, const fw_f32x4 (&acc)[T], uint32_t wave, uint32_t lane) {
#pragma unroll
    for (int t = 0; t < T; ++t) *(fw_f32x4*)(s_sum + ((size_t)(wave * T + t) * 64 + lane) * 4) = acc[t];
}
__device__ __forceinline__ float few_sum(const float* s_sum, uint32_t tiles, uint32_t e, uint32_t waves) { // (four waves or eight, in pairs)
    auto at = [&](uint32_t w) { return s_sum[w * tiles * 256 + e]; };
    const float v = (at(0) + at(1)) + (at(2) + at(3));
    return waves == 4 ? v : v + ((at(4) + at(5)) + (at(6) + at(7)));
}

template <int NB, int MT, int U> __global__ void __launch_bounds__(512) linear_few_kernel(LinearF32Params p) {
    extern __shared__ __attribute__((aligned(16))) float s_sum[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6, r16 = lane & 15, g = lane >> 4;
    const uint32_t n0 = blockIdx.x * 16 * NB, z = blockIdx.z;
    const uint16_t* wp[NB];
    const float* xp[MT];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const uint32_t n = n0 + 16 * j + r16;
        wp[j] = p.w + z * p.w_batch + (size_t)(n < p.n ? n : p.n - 1) * p.k + 8 * g;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const uint32_t r = 16 * i + r16;
        xp[i] = p.x + z * p.x_batch + (size_t)(r < p.rows ? r : p.rows - 1) * p.ldx + 8 * g;
    }
    fw_f32x4 acc[NB][MT] = {};
    few_contract<NB, MT, U>(acc, wp, xp, p.k / kChunk, wave, waves);
    few_put<NB * MT>(s_sum, reinterpret_cast<const fw_f32x4(&)[NB * MT]>(acc), wave, lane);
    __syncthreads();
    float* y = p.y + z * p.y_batch;
    for (uint32_t e = tid; e < NB * MT * 256; e += blockDim.x) {
        const uint32_t t = e >> 8, l = (e >> 2) & 63, row = 16 * (t % MT) + (l & 15), n = n0 + 16 * (t / MT) + 4 * (l >> 4) + (e & 3);
        if (row >= p.rows || n >= p.n) continue;
        y[(size_t)row * p.ldy + n] = linear_epilogue(few_sum(s_sum, NB * MT, e, waves), p.bias ? bf16_to_f32(p.bias[n]) : 0.0f, p, row, z, n);
    }
}

// Experts: a workgroup per expert and tile of its outputs.  The expert's (row, slot) pairs are found in the ids, 16 of them a turn: its weights are read once for all its
// pairs (once per 16), where a workgroup per pair read them again for every one.  GATE: 16 hidden units, gate and up rows, out = act(gate, up) of row pair / top of x; else
// 16 NB outputs of row `pair` of x.  by_slot: fewer pairs than experts, the y index is a pair and the workgroup of the first one with its expert works.
template <bool GATE, int NB>
__global__ void __launch_bounds__(512) experts_few_kernel(const float* x, const int32_t* ids, const uint16_t* w_all, float* out, uint32_t slots, uint32_t k, uint32_t n, uint32_t routed,
                                                          uint32_t top, ExpertAct act, const float* in_weights, uint32_t by_slot) {
    static_assert(!GATE || NB == 2, "a tile of gate and one of up rows");
    extern __shared__ __attribute__((aligned(16))) float s_sum[];
    __shared__ uint16_t s_pair[kFewRowsMaxSlots];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6, r16 = lane & 15, g = lane >> 4;
    const int32_t e = by_slot ? ids[blockIdx.y] : (int32_t)blockIdx.y;
    if (e < 0 || (uint32_t)e >= routed) return; // (uniform over the workgroup, as the next; an identity expert has no weights)
    uint32_t count = 0;
    for (uint32_t base = 0; base < slots; base += 64) { // (every wave finds the same list)
        const bool hit = base + lane < slots && ids[base + lane] == e;
        const unsigned long long m = __ballot(hit);
        if (by_slot && !count && m && base + (uint32_t)__builtin_ctzll(m) != blockIdx.y) return;
        if (hit) s_pair[count + __popcll(m & ((1ull << lane) - 1))] = (uint16_t)(base + lane);
        count += (uint32_t)__popcll(m);
    }
    if (!count) return;
    __syncthreads();
    const uint32_t n0 = blockIdx.x * 16 * (GATE ? 1 : NB);
    const uint16_t* wp[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const uint32_t c = n0 + (GATE ? 0 : 16 * j) + r16, row = (c < n ? c : n - 1) + (GATE && j ? n : 0u);
        wp[j] = w_all + ((size_t)e * (GATE ? 2 : 1) * n + row) * k + 8 * g;
    }
    for (uint32_t c0 = 0; c0 < count; c0 += 16) {
        const uint32_t pair = s_pair[c0 + r16 < count ? c0 + r16 : count - 1];
        const float* xp[1] = {x + (size_t)(GATE ? pair / top : pair) * k + 8 * g};
        fw_f32x4 acc[NB][1] = {};
        few_contract<NB, 1, 2>(acc, wp, xp, k / kChunk, wave, waves);
        if (c0) __syncthreads(); // (the turn before has been read)
        few_put<NB>(s_sum, reinterpret_cast<const fw_f32x4(&)[NB]>(acc), wave, lane);
        __syncthreads();
        for (uint32_t i = tid; i < (GATE ? 1 : NB) * 256; i += blockDim.x) {
            const uint32_t m = c0 + ((i >> 2) & 15), c = n0 + 16 * (i >> 8) + 4 * ((i >> 6) & 3) + (i & 3);
            if (m >= count || c >= n) continue;
            const uint32_t to = s_pair[m];
            float v = few_sum(s_sum, NB, i, waves);
            if (GATE) {
                const float wt = in_weights ? in_weights[to] : 1.0f;
                v = expert_act(wt * few_sum(s_sum, NB, 256 + i, waves), wt * v, act);
            }
            out[(size_t)to * n + c] = v;
        }
    }
}
// y[r] = residual[r] + the row's winners in slot order (identity experts: the block's input itself); y2 [pair][d]
__global__ void __launch_bounds__(256) experts_few_combine_kernel(const float* y2, const float* x, const int32_t* ids, const float* weights, const float* residual, float* y, uint32_t d,
                                                                  uint32_t routed, uint32_t top) {
    const uint32_t r = blockIdx.x, n = blockIdx.y * 256 + threadIdx.x;
    if (n >= d) return;
    float sum = residual ? residual[(size_t)r * d + n] : 0.0f;
    for (uint32_t j = 0; j < top; ++j) {
        const uint32_t pair = r * top + j;
        const int32_t e = ids[pair];
        if (e < 0) continue;
        sum = fmaf(weights ? weights[pair] : 1.0f, (uint32_t)e >= routed ? x[(size_t)r * d + n] : y2[(size_t)pair * d + n], sum);
    }
    y[(size_t)r * d + n] = sum;
}

// waves of a workgroup: eight where the grid has no more than a workgroup per CU and a wave keeps a few chunks of its own, else four (a CU holds one workgroup of eight or
// three of four: 8208 x 2048, 257 workgroups, is 13.8 us with eight)
uint32_t few_waves(size_t workgroups, uint32_t chunks) { return workgroups <= 256 && chunks >= 16 ? 8 : 4; }
template <int NB, int MT, int U> uzu_status launch_few(hipStream_t s, const LinearF32Params& p) {
    const dim3 grid((p.n + 16 * NB - 1) / (16 * NB), 1, p.batch);
    const uint32_t waves = few_waves((size_t)grid.x * p.batch, p.k / kChunk);
    return launch_check([&] { hipLaunchKernelGGL((linear_few_kernel<NB, MT, U>), grid, dim3(64 * waves), (size_t)waves * NB * MT * 1024, s, p); }, "linear_few");
}
} // namespace

// Where it is the faster form.  Up to 16 rows the other one is a wave per column (k_stream32.hip, linear_rows): workgroups of four columns and four rows, 0.25 us + 0.53 us per 1024 k
// for every one a CU gets, against 1.15 us + 0.09 us a row per 1024 k here, whatever the columns.  So narrow outputs and long contractions stay there: 192 x 4096 6.0 us against 8.8 .. 12.7
// (5 .. 16 rows), 512 x 2048 4.7 .. 5.7 against 5.6 .. 7.6, 64 x 1024 3.7 against 3.9 .. 4.9; 1024 x 1024 4.0 .. 5.9 against 4.1 .. 5.1, 2048 x 2048 7.7 .. 12.5 against 5.6 .. 7.5.  One or two
// rows of a wave per column cost no more than their weights' reading (1024 x 1024 2.9 us, 4 here; narrow outputs up to four rows: 3 rows of 2048 x 4096 8.2 us, 8.4 here).
// Above 16 rows the LDS-DMA form (k_linear_mfma.hip) is 12 to 16 us at any of these sizes; here 32 rows are 8.1 us of 1024 x 1024, 13.4 of
// 2048 x 2048, 14.1 of 7712 x 2048, 24 of 8208 x 2048 and of 2048 x 4096.
static bool few_faster(const LinearF32Params& p) {
    const size_t columns = (size_t)p.n * p.batch;
    if (p.rows > 16) return p.k <= 2048 && columns < 8192;
    if (p.rows <= 2 || columns >= 4096) return p.rows > 2;
    if (p.rows <= 4) return false;
    const double k1024 = p.k / 1024.0, a_cu = (double)(((columns + 3) / 4 * ((p.rows + 3) / 4) + 255) / 256);
    return 2.6 + k1024 * (1.15 + 0.088 * p.rows) <= 3.0 + 0.12 * k1024 + a_cu * (0.25 + 0.53 * k1024);
}
bool linear_few_supported(const LinearF32Params& p) {
    return p.bf16_products && p.rows <= 32 && p.k % kChunk == 0 && p.k && few_faster(p) && !p.row_offsets && !p.row_map && p.ldx % 4 == 0 && p.x_batch % 4 == 0 && p.w_batch % 8 == 0 &&
           (((uintptr_t)p.x | (uintptr_t)p.w) & 15) == 0;
}
uzu_status linear_few(hipStream_t s, const LinearF32Params& p) {
    UZU_REQUIRE(linear_few_supported(p), "linear_few: shape / alignment not covered");
    if (p.rows <= 16) return (size_t)p.n * p.batch >= 4096 ? launch_few<2, 1, 2>(s, p) : launch_few<1, 1, 2>(s, p);
    return launch_few<2, 2, 1>(s, p);
}

bool experts_few_supported(const float* x, const float* hidden, const uint16_t* w13, const uint16_t* w2, uint32_t rows, uint32_t d, uint32_t ff, uint32_t routed, uint32_t top, const ExpertAct& act) {
    return rows && routed && routed < 65536 && top && rows * top <= kFewRowsMaxSlots && !act.plain && d % kChunk == 0 && ff % kChunk == 0 && d && ff &&
           (((uintptr_t)x | (uintptr_t)hidden | (uintptr_t)w13 | (uintptr_t)w2) & 15) == 0;
}
template <bool GATE, int NB>
static uzu_status launch_experts_few(hipStream_t s, const float* x, const int32_t* ids, const uint16_t* w, float* out, uint32_t slots, uint32_t k, uint32_t n, uint32_t routed, uint32_t top,
                                     const ExpertAct& act, const float* in_weights) {
    const uint32_t by_slot = slots < routed ? 1u : 0u, tile = 16 * (GATE ? 1 : NB);
    const dim3 grid((n + tile - 1) / tile, by_slot ? slots : routed);
    const uint32_t waves = few_waves((size_t)grid.x * grid.y, k / kChunk);
    return launch_check([&] { hipLaunchKernelGGL((experts_few_kernel<GATE, NB>), grid, dim3(64 * waves), (size_t)waves * NB * 1024, s, x, ids, w, out, slots, k, n, routed, top, act, in_weights, by_slot); },
                        GATE ? "experts_few_gate_up" : "experts_few_down");
}
uzu_status experts_few_gate_up(hipStream_t s, const float* x, const int32_t* ids, const uint16_t* w13, float* hidden, uint32_t rows, uint32_t d, uint32_t ff, uint32_t routed, uint32_t top,
                               const ExpertAct& act, const float* in_weights) {
    return launch_experts_few<true, 2>(s, x, ids, w13, hidden, rows * top, d, ff, routed, top, act, in_weights);
}
uzu_status experts_few_down(hipStream_t s, const float* hidden, const float* x, const int32_t* ids, const float* weights, const uint16_t* w2, const float* residual, float* y2, float* y, uint32_t rows,
                            uint32_t d, uint32_t ff, uint32_t routed, uint32_t top) {
    UZU_PROPAGATE((launch_experts_few<false, 2>(s, hidden, ids, w2, y2, rows * top, ff, d, routed, top, ExpertAct(), nullptr)));
    return launch_check([&] { hipLaunchKernelGGL(experts_few_combine_kernel, dim3(rows, (d + 255) / 256), dim3(256), 0, s, y2, x, ids, weights, residual, y, d, routed, top); }, "experts_few_combine");
}

} // namespace k
} // namespace uzu
