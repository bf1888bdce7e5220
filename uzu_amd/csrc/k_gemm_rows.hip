// k_gemm_rows.hip -- quantised matmul for dozens to hundreds of activation rows: a register-fed matrix-core kernel without operand staging, and for hundreds of rows its staged sibling (below).
//
// Where it sits: behind the few-rows kernel (k_gemv_rows.hip, M <= 16; wide matrices come here from 2 rows on) and in front of the large tiles (k_gemm128.hip).  At these sizes a linear of a 1024-wide
// model is 1 .. 15 GFLOP and 1 .. 4 MB of codes -- a microsecond or two of either -- and what a tile kernel spends is its chain: a k-step of 64 through LDS with
// two barriers is ~1 us whatever else the CU does, so a 64 x 64 tile over K = 3584 was 35 us on sixteen workgroups.  Here nothing is staged and nothing waits:
//   * a wave owns 16 MT tokens x 16 NB weight rows of v_mfma_f32_16x16x32_bf16.  Activations go from the L2 into the A operand (lane (r, g): token r, 16 bytes
//     at k0 + 32 i + 8 g -- an instruction takes whole 64-byte pieces of 16 rows; at k0 + 32 g + 8 i it would touch every piece four times, which is what bounds
//     the cache in front of a CU).  A lane loads 16 bytes = 32 codes of weight row r at k0 + 32 g; four lane swaps (v_permlane32_swap, v_permlane16_swap) turn
//     the (lane group, word) square round, so that word i holds the codes of k0 + 32 i + 8 g, and a word converts to the 8 bf16 (q - 8) / 16 of MFMA i
//     (gemm_convert.h: dequant4).  The codes are centred for the sums' sake: with (16 + q), two codes per v_and_or_b32, partial sums are five times the result and the
//     error against 64 bits is 1.8e-7 of it, here 5e-8 at K = 1024 and 8e-8 at K = 4096 (64 x 64 tiles: 7e-8, 1.4e-7).  The time is the same within 1 %: what the
//     conversion costs more, the activations' permutation to that pair order did;
//   * a step contracts over 128 k = one quant group: the group's products and the tokens' sums (the same A against an all-ones B) are folded with the f32 scale
//     and offset of the lane's own weight row, so no weight is ever rounded and no scalar crosses lanes.  Scales are read two groups at a time;
//   * the next step's loads are in flight while a step is computed, waves never meet before the end, and K is cut KW ways over the waves of a workgroup
//     (added through LDS in wave order) and `splits` ways over workgroups (f32 partial tiles, added in split order by the reduction that also applies the next
//     Normalization): the cuts are chosen so that the chip has a workgroup per CU and a wave's chain is a few steps.
// What bounds it: below ~100 rows the launch and two or three dependent loads; above, the L2 traffic of unshared operands (~7 TB/s at 0.3 PFLOP/s), which the staged kernel shares.
// Measured, us per launch, 64 x 64 tiles -> here (weights not in cache): 1024 x 3584, M = 37: 38.0 -> 8.5; 1024 x 2048: 23.7 -> 6.9; 7168 x 1024 + GatedActMul:
// 14.3 + 4.7 -> 8.1; 8224 x 1024: 14.5 -> 10.3; 4096 x 14336: 163 -> 33; a 37-token prompt of Qwen3.5-0.8B 3.84 -> 2.22 ms.
#include <algorithm>
#include <type_traits>

#include "decode_epilogue.h"
#include "device_utils.h"
#include "gemm_convert.h"
#include "gemm_tile_order.h"
#include "kernels.h"

namespace uzu {
namespace k {

namespace {
typedef __attribute__((ext_vector_type(8))) __bf16 gm_bf16x8;
typedef __attribute__((ext_vector_type(4))) float gm_f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t gm_u32x4;

struct GemmRowsParams {
    const uint16_t* a = nullptr; // [m, k] bf16
    const uint8_t* w = nullptr;  // [n, k / 2]
    const uint16_t* scales = nullptr;
    const uint16_t* biases = nullptr;
    const uint8_t* zp = nullptr;
    const uint16_t* out_bias = nullptr; // [n] or null
    void* d = nullptr;                  // [m, n] (ACT: [m, n / 2]) bf16 or f32
    float* partials = nullptr;          // [splits][m, n] f32, or null: the whole sum is here
    uint32_t m = 0, n = 0, k = 0, d_f32 = 0, act_type = 0, splits = 0;
};

// (lane group g, word j) -> (lane group j, word g): register i of lane group g afterwards holds what word g of lane group i was
__device__ __forceinline__ void turn_words(gm_u32x4& w) {
    typedef __attribute__((ext_vector_type(2))) uint32_t pair;
    pair t = __builtin_bit_cast(pair, __builtin_amdgcn_permlane32_swap(w.x, w.z, false, false));
    w.x = t.x, w.z = t.y;
    t = __builtin_bit_cast(pair, __builtin_amdgcn_permlane32_swap(w.y, w.w, false, false));
    w.y = t.x, w.w = t.y;
    t = __builtin_bit_cast(pair, __builtin_amdgcn_permlane16_swap(w.x, w.y, false, false));
    w.x = t.x, w.y = t.y;
    t = __builtin_bit_cast(pair, __builtin_amdgcn_permlane16_swap(w.z, w.w, false, false));
    w.z = t.x, w.w = t.y;
}

// four consecutive outputs of a token, the whole sums: + bias, f32 or bf16
__device__ __forceinline__ void store_quad(const GemmRowsParams& p, uint32_t token, uint32_t n, gm_f32x4 v) {
    if (p.out_bias) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] += bf16_to_f32(p.out_bias[n + j]);
    }
    if (p.d_f32) {
        *(gm_f32x4*)((float*)p.d + (size_t)token * p.n + n) = v;
        return;
    }
    u32x2_v q;
    q.x = (uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16), q.y = (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
    *(u32x2_v*)((uint16_t*)p.d + (size_t)token * p.n + n) = q;
}

// KW waves of the workgroup's four share a tile and split its steps; the other 4 / KW side by side.  ACT: n = 2 h weight rows [up | gate]; blocks 0 .. NB/2 - 1
// of a wave are up rows, the rest the gate rows of the same outputs, and the epilogue is GatedActMul on the rounded pair.
template <int NB, int MT, int KW, bool ACT, uint32_t KIND> // KIND: uzu_matmul_b_kind (a branch on it in the loop would wait for every load in flight)
__global__ void __launch_bounds__(256, 2) gemm_rows_kernel(GemmRowsParams p) {
    constexpr int OB = ACT ? NB / 2 : NB;   // 16-row blocks of outputs per wave
    constexpr int PITCH = 16 * NB + 4;      // floats per token of a parked tile
    constexpr int GROUPS = 4 / KW;          // tiles side by side in the workgroup
    __shared__ __attribute__((aligned(16))) float s_part[4 * 16 * MT * PITCH];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r = lane & 15, g = lane >> 4, kw = wave % KW, grp_w = wave / KW;
    const uint32_t out_n = ACT ? p.n / 2 : p.n, half_k = p.k / 2, G = p.k / 128, pairs = G / 2;
    const uint32_t row0 = (blockIdx.x * GROUPS + grp_w) * (16 * OB), t0 = blockIdx.y * (16 * MT);
    // this wave's steps, a whole number of pairs (none where there are more waves than pairs: such a wave adds zeros)
    const uint32_t part = blockIdx.z * KW + kw, parts = p.splits * KW;
    const uint32_t s_lo = 2 * (pairs * part / parts), s_hi = 2 * (pairs * (part + 1) / parts);
    // rows and tokens past the end are read from inside the matrices; their sums are never stored
    uint32_t wrow[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const uint32_t base = row0 + 16 * (ACT && b >= OB ? b - OB : b), side = ACT && b >= OB ? out_n : 0u;
        wrow[b] = side + min(base + r, out_n - 1);
    }
    const uint16_t* xrow[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) xrow[t] = p.a + (size_t)min(t0 + 16 * t + r, p.m - 1) * p.k + 8 * g;
    struct Step {
        gm_u32x4 codes[NB], xv[MT][4];
    };
    auto load_step = [&](uint32_t s, Step& st) {
        const uint32_t c = min(s, G - 1); // (a wave without steps)
#pragma unroll
        for (int b = 0; b < NB; ++b) st.codes[b] = *(const gm_u32x4*)(p.w + (size_t)wrow[b] * half_k + 16 * g + (size_t)c * 64);
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) st.xv[t][i] = *(const gm_u32x4*)(xrow[t] + (size_t)c * 128 + 32 * i);
    };
    uint32_t sc2[NB], of2[NB] = {}; // scales / offsets of a pair of groups
    auto load_scales = [&](uint32_t s) {
        const uint32_t c = min(s, G - 2);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const size_t at = (size_t)wrow[b] * G + c;
            sc2[b] = *(const uint32_t*)(p.scales + at);
            if constexpr (KIND == UZU_MATMUL_B_SCALE_BIAS) of2[b] = *(const uint32_t*)(p.biases + at);
            else if constexpr (KIND == UZU_MATMUL_B_SCALE_ZERO_POINT) of2[b] = p.zp[at / 2];
        }
    };
    uint32_t ones = 0x3F803F80u;
    asm("" : "+v"(ones));
    const gm_u32x4 ones4 = {ones, ones, ones, ones};
    gm_f32x4 acc[NB][MT]; // tokens 4 g + v of tile t, row r of block b
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[b][t] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](Step& st, const float (&sc)[NB], const float (&of)[NB]) {
        gm_f32x4 dq[NB][MT], dx[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            dx[t] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int b = 0; b < NB; ++b) dq[b][t] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) turn_words(st.codes[b]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (KIND != UZU_MATMUL_B_SCALE_SYMMETRIC) {
#pragma unroll
                for (int t = 0; t < MT; ++t) dx[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gm_bf16x8, st.xv[t][i]), __builtin_bit_cast(gm_bf16x8, ones4), dx[t], 0, 0, 0);
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const u32x4_t wv = dequant4(st.codes[b][i] ^ 0x88888888u); // (nibbles as two's complement of q - 8)
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    dq[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gm_bf16x8, st.xv[t][i]), __builtin_bit_cast(gm_bf16x8, wv), dq[b][t], 0, 0, 0);
            }
        }
        // group fold: acc += 16 scale dq + (offset + 8 scale) sum_x   (dq = sum (q - 8) / 16 x; a symmetric matrix has nothing left to add)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[b][t][v] = fmaf(sc[b], dq[b][t][v], KIND == UZU_MATMUL_B_SCALE_SYMMETRIC ? acc[b][t][v] : fmaf(of[b], dx[t][v], acc[b][t][v]));
    };
    auto offset_of = [&](float sc, float raw) { // raw: the bf16 offset, or the zero point
        return KIND == UZU_MATMUL_B_SCALE_BIAS ? fmaf(8.0f, sc, raw) : KIND == UZU_MATMUL_B_SCALE_ZERO_POINT ? sc * (8.0f - raw) : 0.0f;
    };
    Step stA, stB;
    load_step(s_lo, stA);
    load_scales(s_lo);
    for (uint32_t s = s_lo; s < s_hi; s += 2) {
        float sc0[NB], of0[NB], sc1[NB], of1[NB];
        load_step(s + 1, stB);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            constexpr bool zp = KIND == UZU_MATMUL_B_SCALE_ZERO_POINT;
            sc0[b] = bits_to_f32(sc2[b] << 16), sc1[b] = bits_to_f32(sc2[b] & 0xFFFF0000u);
            of0[b] = offset_of(sc0[b], zp ? (float)(of2[b] & 15u) : bits_to_f32(of2[b] << 16));
            of1[b] = offset_of(sc1[b], zp ? (float)((of2[b] >> 4) & 15u) : bits_to_f32(of2[b] & 0xFFFF0000u));
            sc0[b] *= 16.0f, sc1[b] *= 16.0f;
        }
        // (a wave of four has two steps of K = 1024: reloads past its end, though nobody waited for them, were a third of what it asked of the L2.  37 rows: 8224 x 1024 11.2 us -> 8.8, 7168 x 1024
        // + GatedActMul 9.3 -> 8.4, 3072 x 1024 7.0 -> 5.6, 1024 x 2048 and x 3584 in four shares 5.6 -> 5.1; 1600 products of 17 .. 128 rows 1.06x on the average.  17 rows of K = 2560 and 3584 lose
        // 1 %, 6144 x 3584 9.2 -> 9.9; a last pair of steps without loads behind a loop with them gives that back, and takes 8 % of every product of K = 512: more code to fetch)
        if (s + 2 < s_hi) load_scales(s + 2);
        __builtin_amdgcn_sched_barrier(0); // (left alone, the scheduler sinks the loads to their uses and waits for each)
        compute(stA, sc0, of0);
        __builtin_amdgcn_sched_barrier(0);
        if (s + 2 < s_hi) load_step(s + 2, stA);
        __builtin_amdgcn_sched_barrier(0);
        compute(stB, sc1, of1);
        __builtin_amdgcn_sched_barrier(0);
    }
    // the tile to LDS by token, waves' shares added in wave order; consecutive threads take consecutive quads of a token's outputs (n % 4 == 0: a quad is all
    // inside or all outside)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) s_part[((size_t)wave * 16 * MT + 16 * t + 4 * g + v) * PITCH + 16 * b + r] = acc[b][t][v];
    lds_barrier();
    constexpr int QUADS = 4 * OB; // per token
    const uint32_t local = tid % (64 * KW);
    const float* base = s_part + (size_t)grp_w * KW * 16 * MT * PITCH;
    for (uint32_t i = local; i < 16 * MT * QUADS; i += 64 * KW) {
        const uint32_t tl = i / QUADS, quad = i % QUADS, token = t0 + tl, n = row0 + 4 * quad;
        if (token >= p.m || n >= out_n) continue;
        const float* at = base + (size_t)tl * PITCH + 4 * quad;
        gm_f32x4 v = *(const gm_f32x4*)at, gate = v;
        if (ACT) gate = *(const gm_f32x4*)(at + 16 * OB);
#pragma unroll
        for (int w = 1; w < KW; ++w) {
            v += *(const gm_f32x4*)(at + (size_t)w * 16 * MT * PITCH);
            if (ACT) gate += *(const gm_f32x4*)(at + (size_t)w * 16 * MT * PITCH + 16 * OB);
        }
        if (p.partials) {
            *(gm_f32x4*)(p.partials + ((size_t)blockIdx.z * p.m + token) * p.n + n) = v;
            continue;
        }
        if (!ACT) {
            store_quad(p, token, n, v);
            continue;
        }
        uint16_t o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) { // the rounded pair the unfused kernels would have stored (gated_act_mul/mod.rs:5-12)
            if (p.out_bias) v[j] += bf16_to_f32(p.out_bias[n + j]), gate[j] += bf16_to_f32(p.out_bias[out_n + n + j]);
            o[j] = f32_to_bf16(round_bf16(round_bf16(v[j]) * act_bf16(p.act_type, round_bf16(gate[j]), kExp2fTab)));
        }
        u32x2_v q;
        q.x = (uint32_t)o[0] | ((uint32_t)o[1] << 16), q.y = (uint32_t)o[2] | ((uint32_t)o[3] << 16);
        *(u32x2_v*)((uint16_t*)p.d + (size_t)token * out_n + n) = q;
    }
}

// ---- hundreds of rows: the same arithmetic, 64 tokens x 128 weight rows a workgroup, operands staged by LDS DMA.
// Four register-fed waves on a tile of 32 x 64 read every operand for themselves, 344 KB a workgroup and 3584 k, and the L2 bounds them (4.7 TB/s).  Here rows, codes, scales and
// offsets of a quant group (26 KB) come by global_load_lds into a ring of three stages, two on their way, and one barrier a group; a wave converts 32 weight rows for all 64 tokens (the A
// operands from LDS), so a code is converted once a workgroup.  What bounds it: vector instructions (240 a wave and group: 112 of the conversion, 64 of the fold) and MFMAs (36) hardly
// overlap, 0.66 us a group with two workgroups a CU, 1.0 with one.  Tried: a wave's activation sums for itself (48 MFMAs) or all tiles' (here: one's, the others' from LDS) and slots
// keyed to the row alone (3 of 7 LDS cycles conflicts): 2 to 3 % each; partials by non-temporal stores: 2 us off here, 1 to 4 us more in whoever reads them.
constexpr int ST = 64, SN = 128; // tokens, weight rows of a staged tile
struct StagedShape {
    static constexpr uint32_t A_BYTES = ST * 256, W_BYTES = SN * 64, S_BYTES = 4 * 256, O_BYTES = 4 * 256, STAGE = A_BYTES + W_BYTES + S_BYTES + O_BYTES, STAGES = 3;
    static constexpr int PITCH = SN + 4; // floats per token of the parked tile
};
static_assert(ST * StagedShape::PITCH * 4 <= StagedShape::STAGE * StagedShape::STAGES, "the parked tile takes the stages' place");

template <uint32_t KIND>
__global__ void __launch_bounds__(256, 2) gemm_rows_staged_kernel(GemmRowsParams p) {
    using S = StagedShape;
    constexpr int OPS = KIND == UZU_MATMUL_B_SCALE_SYMMETRIC ? 7 : 8; // wave-instructions of a stage
    __shared__ __attribute__((aligned(1024))) uint8_t smem[S::STAGE * S::STAGES];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r = lane & 15, g = lane >> 4, G = p.k / 128;
    uint32_t m_t, n_t;
    if (!tile_of_block(blockIdx.x, (p.m + ST - 1) / ST, (p.n + SN - 1) / SN, &m_t, &n_t)) return;
    const uint32_t t0 = m_t * ST, row0 = n_t * SN;
    const uint32_t g_lo = G * blockIdx.y / p.splits, T = G * (blockIdx.y + 1) / p.splits - g_lo;
    // where this lane's pieces come from (rows and tokens past the end: from inside the matrices, never stored).  The 16-byte chunk x of a staged row lies in slot x ^ key(row): the 16 rows
    // that a quarter-wave reads fall on different banks, 256 bytes wide together
    auto a_key = [](uint32_t row) { return row >> 2 | (row & 3) << 2; };
    auto w_key = [](uint32_t row) { return (0u - (row >> 2)) & 3u; };
    uint32_t va[4], vw[2], vs;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t row = wave * 16 + i * 4 + lane / 16;
        va[i] = min(row, p.m - 1 - t0) * p.k * 2 + ((lane & 15) ^ a_key(row & 15)) * 16;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t row = wave * 32 + i * 16 + lane / 4;
        vw[i] = min(row0 + row, p.n - 1) * (p.k / 2) + ((lane & 3) ^ w_key(row & 15)) * 16;
    }
    vs = min(row0 + wave * 32 + (lane & 31), p.n - 1) * G; // (two lanes bring the same)
    const uint8_t* a_base = (const uint8_t*)(p.a + (size_t)t0 * p.k);
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    auto dma16 = [&](const void* base, uint32_t v, uint32_t dst) {
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %0" : : "s"(base), "s"(dst), "v"(v) : "memory", "m0");
    };
    auto fetch = [&](uint32_t t, uint32_t buf) {
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + buf * S::STAGE), grp = g_lo + t;
#pragma unroll
        for (int i = 0; i < 4; ++i) dma16(a_base + (size_t)grp * 256, va[i], dst + (wave * 4 + i) * 1024);
#pragma unroll
        for (int i = 0; i < 2; ++i) dma16(p.w + (size_t)grp * 64, vw[i], dst + S::A_BYTES + (wave * 2 + i) * 1024);
        const uint32_t at = (vs + grp) & ~1u, s_dst = dst + S::A_BYTES + S::W_BYTES + wave * 256; // (G is even: the aligned pair of groups)
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, %0" : : "s"(p.scales), "s"(s_dst), "v"(at * 2) : "memory", "m0");
        if constexpr (KIND == UZU_MATMUL_B_SCALE_BIAS) asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, %0" : : "s"(p.biases), "s"(s_dst + S::S_BYTES), "v"(at * 2) : "memory", "m0");
        else if constexpr (KIND == UZU_MATMUL_B_SCALE_ZERO_POINT)
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_ubyte %2, %0" : : "s"(p.zp), "s"(s_dst + S::S_BYTES), "v"(at / 2) : "memory", "m0");
    };
    // wave w alone sums the activations of token tile w (against an all-ones B) and hands the sums to the others through LDS
    __shared__ __attribute__((aligned(16))) float s_sum[2][ST];
    constexpr bool SUMS = KIND != UZU_MATMUL_B_SCALE_SYMMETRIC;
    const uint32_t w_at = S::A_BYTES + (wave * 32 + r) * 64 + (g ^ w_key(r)) * 16, s_at = S::A_BYTES + S::W_BYTES + wave * 256 + r * 4;
    uint32_t a_at[4]; // MFMA i contracts k = 32 g + 8 i .. of the group in lane group g: word i of the lane's codes as they lie
#pragma unroll
    for (int i = 0; i < 4; ++i) a_at[i] = r * 256 + ((4 * g + i) ^ a_key(r)) * 16;
    gm_u32x4 af[4][4], raw[2], wv[2][2];
    uint32_t sraw[2], oraw[2] = {0u, 0u};
    auto rows = [&](const uint8_t* st, int i) {
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) af[i][tt] = *(const gm_u32x4*)(st + a_at[i] + tt * 4096);
    };
    gm_u32x4 own[4]; // the wave's own tile
    auto own_rows = [&](const uint8_t* st) {
        if constexpr (SUMS)
#pragma unroll
            for (int i = 0; i < 4; ++i) own[i] = *(const gm_u32x4*)(st + a_at[i] + wave * 4096);
    };
    auto codes = [&](const uint8_t* st) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            raw[b] = *(const gm_u32x4*)(st + w_at + b * 1024);
            sraw[b] = *(const uint32_t*)(st + s_at + b * 64);
            if constexpr (SUMS) oraw[b] = *(const uint32_t*)(st + s_at + S::S_BYTES + b * 64);
        }
    };
    auto convert = [&](int i) {
#pragma unroll
        for (int b = 0; b < 2; ++b) wv[i & 1][b] = dequant4(raw[b][i] ^ 0x88888888u);
    };
    uint32_t ones = 0x3F803F80u;
    asm("" : "+v"(ones));
    const gm_u32x4 ones4 = {ones, ones, ones, ones};
    gm_f32x4 acc[2][4], dq[2][4], sums[4]; // dq: a group's products
    float sc[2] = {0.f, 0.f}, of[2] = {0.f, 0.f};
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) acc[0][tt] = acc[1][tt] = dq[0][tt] = dq[1][tt] = sums[tt] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
    auto read_sums = [&](uint32_t which) {
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) sums[tt] = *(const gm_f32x4*)(s_sum[which] + 16 * tt + 4 * g);
    };
    auto fold = [&](int b, int tt) { // acc += 16 scale dq + (offset + 8 scale) sum_x
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[b][tt][v] = fmaf(sc[b], dq[b][tt][v], SUMS ? fmaf(of[b], sums[tt][v], acc[b][tt][v]) : acc[b][tt][v]);
    };

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the counts below are the DMA's alone
    fetch(0, 0);
    if (T > 1) fetch(1, 1);
    uint32_t buf = 0;
    // stage t has landed and every wave has read stage t - 1, whose place stage t + 2 takes
    auto enter = [&](uint32_t t) {
        __builtin_amdgcn_sched_barrier(0);
        if (t + 1 < T) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(OPS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (t + 2 < T) fetch(t + 2, buf == 0 ? 2 : buf - 1);
        __builtin_amdgcn_sched_barrier(0);
    };
    // MFMAs with the vector instructions between them (left alone, the scheduler puts a step's conversions in front of its MFMAs, and the wave's matrix core waits)
    auto interleave = [&](auto mfmas, auto valu) {
#pragma unroll
        for (int i = 0; i < decltype(mfmas)::value; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, decltype(valu)::value, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    enter(0);
    codes(smem), rows(smem, 0), rows(smem, 1), own_rows(smem), convert(0);
    for (uint32_t t = 0; t < T; ++t) {
        const uint8_t* st = smem + buf * S::STAGE;
        const gm_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        const bool hi = (g_lo + t) & 1;
        float nsc[2], nof[2] = {0.f, 0.f};
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const float s = bits_to_f32(hi ? sraw[b] & 0xFFFF0000u : sraw[b] << 16);
            if constexpr (KIND == UZU_MATMUL_B_SCALE_BIAS) nof[b] = fmaf(8.0f, s, bits_to_f32(hi ? oraw[b] & 0xFFFF0000u : oraw[b] << 16));
            else if constexpr (KIND == UZU_MATMUL_B_SCALE_ZERO_POINT) nof[b] = s * (8.0f - (float)((oraw[b] >> (hi ? 4 : 0)) & 15u));
            nsc[b] = s * 16.0f;
        }
        gm_f32x4 dx = zero;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i < 2) rows(st, i + 2);
            if (i < 3) convert(i + 1);
            if (i == 1 && SUMS && r == 0) *(gm_f32x4*)(s_sum[t & 1] + 16 * wave + 4 * g) = dx;
            if (i == 2) { // stage t's operands are in registers
                buf = buf == 2 ? 0 : buf + 1;
                enter(t + 1);
                if constexpr (SUMS) read_sums(t & 1);
                codes(smem + buf * S::STAGE), rows(smem + buf * S::STAGE, 0);
            }
            if (i == 3) rows(smem + buf * S::STAGE, 1);
            if (SUMS && i == 0)
#pragma unroll
                for (int j = 0; j < 4; ++j) dx = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gm_bf16x8, own[j]), __builtin_bit_cast(gm_bf16x8, ones4), dx, 0, 0, 0);
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    if (i == 0) fold(b, tt); // the group before
                    dq[b][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gm_bf16x8, af[i][tt]), __builtin_bit_cast(gm_bf16x8, wv[i & 1][b]), i ? dq[b][tt] : zero, 0, 0, 0);
                }
            if (i == 3) own_rows(smem + buf * S::STAGE), convert(0);
            if (i == 0) interleave(std::integral_constant<int, SUMS ? 12 : 8>(), std::integral_constant<int, 8>());
            else interleave(std::integral_constant<int, 8>(), std::integral_constant<int, 4>());
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) sc[b] = nsc[b], of[b] = nof[b];
    }
    lds_barrier(); // (the reads beyond the last stage) the stages are free
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) fold(0, tt), fold(1, tt);
    float* s_tile = (float*)smem;
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) s_tile[(16 * tt + 4 * g + v) * S::PITCH + wave * 32 + 16 * b + r] = acc[b][tt][v];
    lds_barrier();
#pragma unroll
    for (int i = 0; i < ST * SN / 4 / 256; ++i) {
        const uint32_t at = i * 256 + tid, token = t0 + at / (SN / 4), n = row0 + at % (SN / 4) * 4;
        if (token >= p.m || n >= p.n) continue;
        gm_f32x4 v = *(const gm_f32x4*)(s_tile + at / (SN / 4) * S::PITCH + at % (SN / 4) * 4);
        if (p.partials) *(gm_f32x4*)(p.partials + ((size_t)blockIdx.y * p.m + token) * p.n + n) = v;
        else store_quad(p, token, n, v);
    }
}

struct GemmRowsPlan {
    int nb, kw;
    uint32_t splits, workgroups;
    bool staged;
};

uint32_t staged_tiles(const MatmulParams& p) { return ((p.m + ST - 1) / ST) * ((p.n + SN - 1) / SN); }
bool staged_fits(const MatmulParams& p) { return p.m >= 128 && !p.act_mul && (uint64_t)p.n * p.k / 2 < (1ull << 32) && (uint64_t)ST * p.k * 2 < (1ull << 32); } // (32-bit offsets)

// The cuts: 16-row blocks per wave, waves per tile, K splits over workgroups.  A launch wants about a workgroup per CU; narrow problems take two blocks per wave,
// then all four waves on one tile, then splits (measured at N 1024 .. 8224, K 1024 .. 3584, M 20 .. 1021).
GemmRowsPlan gemm_rows_plan(const MatmulParams& p, int num_cus, bool shares_fit = true) { // (no shares of K over workgroups where there is no room for their sums)
    GemmRowsPlan q{};
    const uint32_t blocks = ((p.act_mul ? p.n / 2 : p.n) + 15) / 16, token_tiles = (p.m + 31) / 32, pairs = p.k / 256, cus = (uint32_t)num_cus;
    auto tiles = [&](uint32_t nb) { const uint32_t ob = p.act_mul ? nb / 2 : nb; return ((blocks + ob - 1) / ob) * token_tiles; };
    const bool long_k = p.k >= 8192; // enough steps to split four-block tiles as well (4096 x 14336, M = 48: 42 -> 33 us)
    q.nb = tiles(2) <= (long_k ? cus / 2 : cus) ? 2 : 4;
    const uint32_t t = tiles(q.nb);
    q.kw = t <= cus + cus / 4 ? 4 : t <= 2 * cus + cus / 2 ? 2 : 1;
    q.splits = 1;
    // shares of K over workgroups from K = 2048 on (below, a share's launch of its own costs more than the steps it takes off: 1024 x 1024 5.7 us whole, 6.2 in two shares, 1024 x 1536 6.7
    // and 7.0), at the most two pairs for a share's waves together: 1024 x 2048 6.9 in four, 8.5 in two; 1024 x 3072 7.7 and 9.1 in two; 512 x 3584 8.3 and 9.4 in two (33 rows)
    if (shares_fit && !p.act_mul && (q.nb == 2 || long_k) && pairs >= 8)
        while (q.splits * 2 * t <= cus && q.splits * 4 <= pairs) q.splits *= 2;
    const uint32_t side_by_side = 4 / q.kw, ob = p.act_mul ? q.nb / 2 : q.nb;
    q.workgroups = ((blocks + ob * side_by_side - 1) / (ob * side_by_side)) * token_tiles * q.splits;
    if (!staged_fits(p)) return q;
    // From 128 rows on the staged kernel may be the faster one; both in us, fitted to 68 sizes of 128 to 640 rows (the worst choice among them costs 1.3 us).  Register-fed: 4 + 15 per 1024 k over the waves
    // and shares that walk it, a begun round 0.9 of a full one.  Staged: 4.5 + 1.0 a group of its share while there is at most one workgroup a CU, 6 + 1.43 for two, and in proportion
    // beyond.  Shares cost what writing the partial tiles takes, and a launch to add them unless the Normalization behind does.
    // us, register-fed -> staged: 517 x 1024 x 2048 18.1 -> 13.0 (three shares), x 3584 23.2 -> 16.0; 517 x 2048 x 1024 16.4 -> 12.4, x 3072 18.0 -> 12.7, x 4096 27.3 -> 16.9; 256 x 8224 x 1024
    // 32.5 -> 16.8; 256 x 4096 x 8192 62.6 -> 37.6 + 5; the other way round 128 x 1024 x 1024 5.8 and 8.3, 256 x 1024 x 2048 8.8 and 10.8, 384 x 1024 x 1024 7.7 and 9.4.
    const bool norm = p.post_norm && p.post_norm_done;
    auto shares = [&](uint32_t splits) { const double mb = 4e-6 * p.m * p.n * splits; return splits == 1 ? 0.0 : mb / 3 + (norm ? mb / 8 : 2.5 + mb / 4); };
    const uint32_t full = q.workgroups / cus, rest = q.workgroups % cus;
    double best = 4.0 + p.k / 1024.0 * 15.0 / (q.kw * q.splits) * (q.nb / 4.0) * (!rest ? full : full ? full + 0.9 : 1.0) + shares(q.splits);
    // (an XCD has an eighth of a share's tiles, rounded up: 400 x 768 x 3584 in six shares of 42 tiles, 36 workgroups on some XCDs' 32 CUs, 17.9 us, in five 15.4)
    const uint32_t staged = staged_tiles(p), groups = p.k / 128, xcd_cus = std::max(cus / 8, 1u);
    for (uint32_t splits = 1; splits <= (shares_fit ? 16u : 1u) && 2 * splits <= groups; ++splits) {
        const uint32_t each = (groups + splits - 1) / splits, per_cu = ((staged + 7) / 8 * splits + xcd_cus - 1) / xcd_cus;
        const double us = (per_cu == 1 ? 4.5 + each : 6.0 + 0.715 * each * per_cu) + shares(splits);
        if (us < best) best = us, q.staged = true, q.splits = splits, q.workgroups = staged * splits;
    }
    return q;
}

template <int NB, int MT, int KW, bool ACT> uzu_status launch_gr(hipStream_t s, const GemmRowsParams& q, uint32_t kind) {
    const uint32_t out_n = ACT ? q.n / 2 : q.n, per = 16 * (ACT ? NB / 2 : NB) * (4 / KW);
    const dim3 grid((out_n + per - 1) / per, (q.m + 16 * MT - 1) / (16 * MT), q.splits);
    switch (kind) {
    case UZU_MATMUL_B_SCALE_BIAS: return launch_check([&] { hipLaunchKernelGGL((gemm_rows_kernel<NB, MT, KW, ACT, UZU_MATMUL_B_SCALE_BIAS>), grid, dim3(256), 0, s, q); }, "gemm_rows");
    case UZU_MATMUL_B_SCALE_ZERO_POINT: return launch_check([&] { hipLaunchKernelGGL((gemm_rows_kernel<NB, MT, KW, ACT, UZU_MATMUL_B_SCALE_ZERO_POINT>), grid, dim3(256), 0, s, q); }, "gemm_rows");
    default: return launch_check([&] { hipLaunchKernelGGL((gemm_rows_kernel<NB, MT, KW, ACT, UZU_MATMUL_B_SCALE_SYMMETRIC>), grid, dim3(256), 0, s, q); }, "gemm_rows");
    }
}
uzu_status launch_staged(hipStream_t s, const GemmRowsParams& q, uint32_t kind) {
    const dim3 grid(tile_order_grid((q.m + ST - 1) / ST, (q.n + SN - 1) / SN), q.splits);
    switch (kind) {
    case UZU_MATMUL_B_SCALE_BIAS: return launch_check([&] { hipLaunchKernelGGL(gemm_rows_staged_kernel<UZU_MATMUL_B_SCALE_BIAS>, grid, dim3(256), 0, s, q); }, "gemm_rows_staged");
    case UZU_MATMUL_B_SCALE_ZERO_POINT: return launch_check([&] { hipLaunchKernelGGL(gemm_rows_staged_kernel<UZU_MATMUL_B_SCALE_ZERO_POINT>, grid, dim3(256), 0, s, q); }, "gemm_rows_staged");
    default: return launch_check([&] { hipLaunchKernelGGL(gemm_rows_staged_kernel<UZU_MATMUL_B_SCALE_SYMMETRIC>, grid, dim3(256), 0, s, q); }, "gemm_rows_staged");
    }
}
template <int NB, int MT, bool ACT> uzu_status launch_kw(hipStream_t s, const GemmRowsParams& q, uint32_t kind, int kw) {
    return kw == 1 ? launch_gr<NB, MT, 1, ACT>(s, q, kind) : kw == 2 ? launch_gr<NB, MT, 2, ACT>(s, q, kind) : launch_gr<NB, MT, 4, ACT>(s, q, kind);
}

bool gemm_rows_supported(const MatmulParams& p) {
    if (exact_mode() || p.m < 2 || p.m > 65535 || p.bits != 4 || p.b_kind == UZU_MATMUL_B_FULL_PRECISION) return false;
    if (p.w_dt != UZU_BF16 || p.a_dt != UZU_BF16 || (p.d_dt != UZU_BF16 && p.d_dt != UZU_F32)) return false;
    if (p.signed_codes || p.ab_scale != 1.0f || p.accumulate || p.has_soft_cap || p.gather) return false;
    if (p.act_mul ? (p.n % 8 || p.d_dt != UZU_BF16) : p.n % 4) return false; // whole quads of outputs
    if (p.group_size != 128 || p.k % 256) return false; // scales and offsets are read two groups at a time
    if (((uintptr_t)p.scales | (uintptr_t)p.biases) & 3) return false;
    return (((uintptr_t)p.a | (uintptr_t)p.b | (uintptr_t)p.d) & 15) == 0;
}

} // namespace

// Where this kernel is the faster one, from measurements of 23 matrices at 2 to 16 rows, of 33 at 20 to 127 and of 24 at 128 to 2043.
//   * Up to 16 rows the other choice is the few-rows kernel (k_gemv_rows.hip), a workgroup per 16 outputs: 1024 x 3584 in 5.6 us against 6.8 here at 5 rows, but 248320 x 1024
//     in 67 .. 125 us (2 .. 16 rows) against 46 .. 53, 4096 x 14336 in 25 .. 28 against 16 .. 20, 28672 x 4096 in 28 .. 44 against 28 .. 30, 8224 x 1024 in 7.2 against 6.0
//     (13 rows).  It also is the better one where a round of workgroups here leaves CUs idle: 34816 x 5120 with GatedActMul (272 workgroups) 40 .. 57 against 53 .. 64,
//     22016 x 2048 with it (172) 12 .. 16 against 15 .. 17, 12288 x 4096 (192) 12.4 against 13.8 at 2 rows; from 8 rows on 15.6 .. 20 against 14.8 .. 15.7.
//   * Up to 19 rows there is none but the GEMV (28672 x 4096, 17 rows: 171 us against 30).
//   * Up to 127 rows it is the 64 x 64 tile (k_gemm.hip), with GatedActMul as a launch of its own behind it.  A tile walks 1024 k in 10.5 us while there is one a CU, in 12.3 while
//     there are two, then in 4 + 5 a tile of a CU's share.  Here a round of workgroups walks 1024 k in 15 us / waves on a tile / splits, and a round that begins with fewer workgroups than
//     CUs costs 0.7 of a full one (the workgroups share what the CU reads).  14336 x 4096: 45.6 us against 32.9 at 64 rows, 53 against 60 at 96; 22016 x 2048 with GatedActMul
//     43 against 66 at 96 rows; 57344 x 8192 with it 217 against 220 at 48, 336 against 465 at 127; 8192 x 8192 86 against 60 at 127.  The slower one is
//     taken at 5 of 264 sizes by more than 3 %, the worst 16 % (18944 x 3584 at 33 rows, 44.6 against 38.6).
//   * From 128 rows on it is the 128 x 128 tile (k_gemm128.hip).  The staged kernel is ahead while its tiles leave a CU free, at every K below 8192 (us, all launches of a product, large tile
// against here): 1021 x 1024 x 2048 26.1 and 20.2, x 3584 38.6 and 28.3, x 7168 48.4 and 36.1; 448 x 4096 x 2048 35.4 and 21.5, x 4096 46.0 and 37.5; 300 x 6144 x 2048 40.0 and 21.6,
// x 7168 89.0 and 58.6; 1021 x 1920 x 1024 27.3 and 13.8; 1900 x 1024 x 1536 28.3 and 17.5.  Beyond, and where GatedActMul is in it, by the work: at 517 x 8224 x 1024 the large tile takes 24.6, the
// staged one 26.7; 1024 rows of 4096 x 512 14.8 and 19.3 (register-fed), 300 x 8192 x 256 11.7 and 12.4.
// From K = 8192 on a workgroup a CU here walks K in 4 us per 1024 and as often as the tiles go round; the large tiles take 12 us and 14 us per 1024 of their share of K, where the
// number of quant groups lets it be cut: 4096 x 8192 46 us against 33 at M = 128 (one round), 48 against 62 at M = 160 (two); 2048 x 11008, which cannot be cut, 150 against
// 41 at M = 256, 150 against 74 at M = 512, 4096 x 9728 (two shares) 82 against 62 at M = 256, 85 against 117 at M = 288; 4096 x 14336 74 against 53 at M = 128, 77 against 101 at
// M = 256; 2048 x 16384 77 against 60 at M = 256, 81 against 118 at M = 288.
bool gemm_rows_preferred(const MatmulParams& p, int num_cus) {
    if (!gemm_rows_supported(p) || (p.m >= 128 && (tune_env("gemm_form") || tune_env("gemm_splits")))) return false; // (a pinned form or split-K is the large tile's)
    const uint32_t cus = (uint32_t)num_cus;
    if (p.m < 128) {
        const GemmRowsPlan plan = gemm_rows_plan(p, num_cus);
        const uint32_t full = plan.workgroups / cus, rest = plan.workgroups % cus, filled = rest ? full + 1 : full;
        if (p.m <= 16) {
            if ((uint64_t)p.n * p.k < (32u << 20)) return p.m > 8 && p.n >= 8192;
            return p.k >= 8192 || (p.m > 4 && !p.act_mul) || 4 * plan.workgroups > 3 * filled * cus;
        }
        if (p.m < 20) return true;
        const double k1024 = p.k / 1024.0, tiles_per_cu = (double)((p.m + 63) / 64) * ((p.n + 63) / 64) / cus;
        const double here = k1024 * 15.0 / (plan.kw * plan.splits) * (plan.nb / 4.0) * (!rest ? full : full ? full + 0.7 : 1.0);
        const double tile = k1024 * (tiles_per_cu <= 1.0 ? 10.5 : std::max(12.3, 4.0 + 5.0 * tiles_per_cu)) + (p.act_mul ? 2.0 + 1.5e-6 * p.m * p.n : 0.0);
        return here <= tile;
    }
    const uint32_t large_tiles = ((p.m + 127) / 128) * ((p.n + 127) / 128);
    if (p.k < 8192) return (staged_fits(p) && staged_tiles(p) < cus) || (2e-9 * p.m * p.n * p.k <= 4.5 && large_tiles < cus * 3 / 4);
    const uint32_t splits = gemm128_splits(p, num_cus), rounds = (((p.n + 63) / 64) * ((p.m + 31) / 32) + cus - 1) / cus;
    if (!splits) return true;
    const uint32_t large_rounds = (large_tiles * splits + cus - 1) / cus;
    return 4ull * p.k * rounds <= 12 * 1024 + 14ull * (p.k / splits) * large_rounds;
}

// host arithmetic only: the cuts of K over workgroups and the grid
void gemm_rows_plan_query(const MatmulParams& p, int num_cus, uint32_t* splits, uint32_t* workgroups) {
    const GemmRowsPlan plan = gemm_rows_plan(p, num_cus);
    *splits = plan.splits, *workgroups = plan.workgroups;
}

uzu_status gemm_rows(hipStream_t s, const MatmulParams& p, int num_cus) {
    GemmRowsPlan plan = gemm_rows_plan(p, num_cus);
    GemmRowsParams q{};
    q.a = (const uint16_t*)p.a, q.w = (const uint8_t*)p.b, q.scales = (const uint16_t*)p.scales, q.biases = (const uint16_t*)p.biases, q.zp = p.zero_points;
    q.out_bias = (const uint16_t*)p.bias, q.d = p.d, q.m = p.m, q.n = p.n, q.k = p.k;
    q.d_f32 = p.d_dt == UZU_F32, q.act_type = p.act_type, q.splits = plan.splits;
    const size_t total = (size_t)p.m * p.n;
    if (plan.splits > 1) {
        q.partials = (float*)stream_workspace(s, (size_t)plan.splits * total * 4);
        if (!q.partials) plan = gemm_rows_plan(p, num_cus, false), q.splits = 1; // (a stream under capture has no workspace)
    }
    uzu_status st;
    if (plan.staged) st = launch_staged(s, q, p.b_kind);
    else if (p.act_mul) st = plan.nb == 2 ? launch_kw<2, 2, true>(s, q, p.b_kind, plan.kw) : launch_kw<4, 2, true>(s, q, p.b_kind, plan.kw);
    else st = plan.nb == 2 ? launch_kw<2, 2, false>(s, q, p.b_kind, plan.kw) : launch_kw<4, 2, false>(s, q, p.b_kind, plan.kw);
    if (st != UZU_OK || q.splits == 1) return st;
    return gemm_split_finish(s, p, q.partials, q.splits);
}

} // namespace k
} // namespace uzu
