// k_gemm_dma.hip -- the large-tile prefill product of int4 codes in groups of 128 (k_gemm128.hip's arithmetic, bit for bit) with every operand brought by LDS DMA.
//
// k_gemm128.hip takes the activation tile through vector registers (loads, 16 v_perm, 4 LDS stores a thread and k-step), a quarter of its time.  Here the rows are in memory in the
// pair order of the int4 conversion already (MatmulParams::a_pairs: a copy by the Normalization, the gated epilogue's own rows, or the pre-pass), so tiles, codes and scales go from the
// L2 to LDS by global_load_lds_dwordx4 / dword into a ring of three stages, two of them on their way; nothing but the conversion, the MFMAs and the group fold is left in the loop.
//   * four waves, 128 x 128, 64-deep stages, two workgroups per CU: they cover each other's prologue and epilogue;
//   * eight waves, 128 x 256, 128-deep stages (a group each, one barrier a group), one workgroup per CU: less L2 -> LDS traffic, ahead where K is long.
// The first operands of a stage are read, and its barrier passed, two MFMA steps before the stage before it ends; a block's fold comes right in front of its next MFMA.
// Bound by the vector instructions beside the MFMAs (7.7 each: conversion 4.5, fold 2) and the card's power limit (2.0 .. 2.2 GHz meanwhile): with neither conversion nor fold
// 1005 TFLOP/s.  Measured, us, 4096 rows (register-staged forms -> four waves / eight waves, the pre-pass's copy included): 14336 x 4096 547 -> 540 / 522, 28672 x 4096 with
// GatedActMul 1224 -> 1078 / 1081, 4096 x 14336 581 -> 617 / 537, 6144 x 4096 263 -> 252 / 255; 2048 rows: 8224 x 1024 68 -> 64 / 73, 7168 x 1024 with it 72 -> 66 / 90.
#include "device_utils.h"
#include "gemm128_epilogue.h"
#include "gemm_convert.h"
#include "gemm_tile_order.h"
#include "kernels.h"
#include "uzu_math.h"

namespace uzu {
namespace k {

namespace {

constexpr int DM = 128; // rows of a workgroup tile

// PIECES wave-instructions of 1 KB: from base + v[i] (16 bytes a lane) to dst + 1024 i + 16 lane
template <int PIECES> __device__ __forceinline__ void dma_rows(const void* base, const uint32_t (&v)[PIECES], uint32_t dst) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %0" : : "s"(base), "s"(dst + 1024 * i), "v"(v[i]) : "memory", "m0");
}
__device__ __forceinline__ void dma_dword(const void* base, uint32_t v, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, %0" : : "s"(base), "s"(dst), "v"(v) : "memory", "m0");
}

// NW waves as 2 x NW/2, each 64 x 64; KS 64-deep k-steps per stage
template <int NW> struct DmaShape {
    static constexpr int NWN = NW / 2, KS = NW == 8 ? 2 : 1, STAGES = 3;
    static constexpr uint32_t A_BYTES = DM * 128 * KS, W_BYTES = 64 * NWN * 32 * KS, S_BYTES = NW * 256, STAGE = A_BYTES + W_BYTES + S_BYTES;
    static constexpr int AP = A_BYTES / 1024 / NW, WP = W_BYTES / 1024 / NW, OPS = AP + WP + 1; // wave-instructions of a stage
};

} // namespace

template <int NW>
__global__ void __launch_bounds__(64 * NW, 2) gemm_q4_dma_kernel(MatmulParams p, const uint16_t* ap, const float* rowsum, const float* coef, float* partials) {
    using S = DmaShape<NW>;
    constexpr int NWN = S::NWN, KS = S::KS, AP = S::AP, WP = S::WP;
    constexpr uint32_t AROW = 128 * KS, ACH = AROW / 16, WROW = 32 * KS, WCH = WROW / 16;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[S::STAGE * S::STAGES];
    __shared__ uint64_t s_exp_tab[32]; // gated epilogue only
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / NWN, wn = wave % NWN, h = lane >> 5, c = lane & 31;
    const uint32_t M = p.m, N = p.n, K = p.k, G = K / 128;
    const bool gated = p.act_mul != 0;
    const uint32_t H = N / 2, m_tiles = (M + DM - 1) / DM, n_tiles = gated ? (H + 32 * NWN - 1) / (32 * NWN) : (N + 64 * NWN - 1) / (64 * NWN);
    uint32_t m_t, n_t;
    if (!tile_of_block(blockIdx.x, m_tiles, n_tiles, &m_t, &n_t)) return;
    const uint32_t m0 = m_t * DM, n0 = n_t * 64 * NWN;
    const uint32_t z = blockIdx.y, Gz = G / gridDim.y, g_lo = z * Gz;
    const uint32_t flip = p.signed_codes ? 0x88888888u : 0u; // the unsigned code u of bf16(16 + u)
    // matrix row of local column l of the tile; gated: 64-column blocks alternate up, gate
    auto column = [&](uint32_t l) -> uint32_t {
        if (!gated) return min(n0 + l, N - 1);
        return min(n_t * (32 * NWN) + (l >> 7) * 64 + (l & 63), H - 1) + ((l & 64) ? H : 0u);
    };

    // ---- where this lane's pieces come from.  A staged row's 16-byte chunk x lies in slot x ^ key(row); the LDS is 256 bytes of banks wide, so the 16 rows that a quarter-wave
    // reads at one k fall on different banks where the key steps once per 256 bytes of rows
    uint32_t va[AP], vw[WP], vs;
#pragma unroll
    for (int i = 0; i < AP; ++i) {
        const uint32_t row = (wave * AP + i) * (64 / ACH) + lane / ACH, chunk = (lane % ACH) ^ (row / (256 / AROW) & (ACH - 1));
        va[i] = min(row, M - 1 - m0) * K * 2 + chunk * 16;
    }
#pragma unroll
    for (int i = 0; i < WP; ++i) {
        const uint32_t col = (wave * WP + i) * (64 / WCH) + lane / WCH, chunk = (lane % WCH) ^ (col / (256 / WROW) & (WCH - 1));
        vw[i] = column(col) * (K / 2) + chunk * 16;
    }
    uint32_t ncol[2];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) ncol[nb] = column(wn * 64 + nb * 32 + c);
    const uint32_t own = column(wn * 64 + lane) * G; // scales of this lane's column
    vs = 0;
    const uint8_t* a_base = (const uint8_t*)(ap + (size_t)m0 * K) + (size_t)g_lo * 256;
    const uint8_t* w_base = (const uint8_t*)p.b + (size_t)g_lo * 64;
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    const uint32_t T = Gz * (2 / KS); // stages of this workgroup's share of K
    auto fetch = [&](uint32_t t, uint32_t buf) {
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + buf * S::STAGE);
        dma_rows<AP>(a_base + (size_t)t * AROW, va, dst + wave * AP * 1024);
        dma_rows<WP>(w_base + (size_t)t * WROW, vw, dst + S::A_BYTES + wave * WP * 1024);
        vs = ((own + g_lo + (KS == 2 ? t : t >> 1)) & ~1u) * 2; // the aligned pair that holds the group's scale
        dma_dword(p.scales, vs, dst + S::A_BYTES + S::W_BYTES + wave * 256);
    };

    f32x16_t acc_g[2][2], acc_t[2][2];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc_g[mb][nb][r] = 0.f, acc_t[mb][nb][r] = 0.f;

    const uint32_t a_at = (wm * 64 + c) * AROW, a_key = c / (256 / AROW) & (ACH - 1);
    const uint32_t w_at = S::A_BYTES + (wn * 64 + c) * WROW, w_key = c / (256 / WROW) & (WCH - 1);
    const uint32_t s_at = S::A_BYTES + S::W_BYTES + wave * 256 + c * 4;

    // MFMA s of a 64-deep k-step takes k = 8 s .. of the step's first half in lanes 0 .. 31, of its second half in lanes 32 .. 63 (k_gemm128.hip's order)
    u32x4_t raw[2], af[4][2], bf[2][2];
    auto codes = [&](const uint8_t* st, int half) {
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) raw[nb] = *(const u32x4_t*)(st + w_at + nb * 32 * WROW + (((half * 2 + h) ^ w_key) * 16));
    };
    auto rows = [&](const uint8_t* st, int half, int s) {
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) af[s][mb] = *(const u32x4_t*)(st + a_at + mb * 32 * AROW + (((half * 8 + 4 * h + s) ^ a_key) * 16));
    };
    auto convert = [&](int s) {
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) bf[s & 1][nb] = dequant4_pairs(raw[nb][s] ^ flip);
    };
    auto mfma = [&](int s, int mb, int nb, bool first) {
        const f32x16_t zero = {};
        acc_g[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, af[s][mb]), __builtin_bit_cast(bf16x8_t, bf[s & 1][nb]), first ? zero : acc_g[mb][nb], 0, 0, 0);
    };
    float sc[2] = {0.f, 0.f};
    auto fold = [&](int mb, int nb) { // acc_t += scale * acc_g
#pragma unroll
        for (int r = 0; r < 16; r += 2) { // in place through inline asm: the register allocator left to itself moves accumulator tuples around the loop
            float t0 = acc_t[mb][nb][r], t1 = acc_t[mb][nb][r + 1];
            asm volatile("v_fmac_f32_e32 %0, %2, %3\n\tv_fmac_f32_e32 %1, %2, %4" : "+v"(t0), "+v"(t1) : "v"(sc[nb]), "v"(acc_g[mb][nb][r]), "v"(acc_g[mb][nb][r + 1]));
            acc_t[mb][nb][r] = t0, acc_t[mb][nb][r + 1] = t1;
        }
        __builtin_amdgcn_sched_barrier(0); // the block's next MFMA must not be hoisted above its fold
    };

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the counts below are the DMA's alone
    fetch(0, 0);
    if (T > 1) fetch(1, 1);
    uint32_t buf = 0;
    // stage t has landed and every wave has read stage t - 1, whose place stage t + 2 takes
    auto enter = [&](uint32_t t) {
        __builtin_amdgcn_sched_barrier(0);
        if (t + 1 < T) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(S::OPS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (t + 2 < T) fetch(t + 2, buf == 0 ? 2 : buf - 1);
        __builtin_amdgcn_sched_barrier(0);
    };
    enter(0);
    codes(smem, 0), rows(smem, 0, 0), rows(smem, 0, 1), convert(0);
    uint32_t t = 0;
    for (uint32_t g = g_lo; g < g_lo + Gz; ++g) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const uint8_t* st = smem + buf * S::STAGE;
            const int in = KS == 2 ? half : 0; // the k-step's place in its stage
            float nsc[2] = {0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 4; ++s) { // A two MFMA steps ahead, codes converted one ahead; a step's last two MFMA steps bring the next one's first operands
                if (s < 2) rows(st, in, s + 2);
                if (s < 3) convert(s + 1);
                if (s == 2) {
                    if (half == 0 && KS == 2) codes(st, 1), rows(st, 1, 0);
                    else {
                        if (half == 1)
#pragma unroll
                            for (int nb = 0; nb < 2; ++nb) nsc[nb] = bits_to_f32((uint32_t)*(const uint16_t*)(st + s_at + nb * 128 + ((ncol[nb] * G + g) & 1) * 2) << 16);
                        ++t;
                        buf = buf == 2 ? 0 : buf + 1;
                        enter(t);
                        codes(smem + buf * S::STAGE, 0), rows(smem + buf * S::STAGE, 0, 0);
                    }
                }
                if (s == 3) rows(smem + buf * S::STAGE, half == 0 && KS == 2 ? 1 : 0, 1);
#pragma unroll
                for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                    for (int nb = 0; nb < 2; ++nb) {
                        if (half == 0 && s == 0) {
                            if (mb + nb == 0) asm volatile("s_nop 15\n\ts_nop 3"); // (the compiler does not see an MFMA's result read through inline asm)
                            fold(mb, nb);
                        }
                        mfma(s, mb, nb, half == 0 && s == 0);
                    }
                if (s == 3) convert(0);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (half == 1) sc[0] = nsc[0], sc[1] = nsc[1];
        }
    }
    asm volatile("s_nop 15\n\ts_nop 3");
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) fold(mb, nb);
    lds_barrier(); // (the reads beyond the last stage) the stages are free: the epilogue's tiles take their place
    const GemmTile tile{m0 + wm * 64, n0 + wn * 64, n_t * (32 * NWN) + (wn >> 1) * 64, n_t * (NWN / 2) + (wn >> 1), {ncol[0], ncol[1]}, (uint32_t)wave, (uint32_t)wn, M, M, N, H, g_lo, g_lo + Gz, z, gated, !gated || n_t * (32 * NWN) + (wn >> 1) * 64 < H};
    gemm_tile_finish<true>(p, tile, rowsum, coef, partials, acc_t, smem, s_exp_tab);
}

bool gemm_q4_dma_supported(const MatmulParams& p) {
    return p.bits == 4 && p.group_size == 128 && p.k % 128 == 0 && (uintptr_t)p.scales % 4 == 0 && (uintptr_t)p.b % 16 == 0 && (size_t)p.n * (p.k / 128) % 2 == 0 &&
           (uint64_t)DM * p.k * 2 < (1ull << 32) && (uint64_t)p.n * p.k / 2 < (1ull << 32) && p.k >= 256;
}
uint32_t gemm_q4_dma_blocks(uint32_t m, uint32_t n, bool gated, bool wide) {
    const uint32_t m_tiles = (m + DM - 1) / DM, cols = wide ? 256 : 128, n_tiles = gated ? (n / 2 + cols / 2 - 1) / (cols / 2) : (n + cols - 1) / cols;
    return tile_order_grid(m_tiles, n_tiles);
}
uzu_status gemm_q4_dma(hipStream_t s, const MatmulParams& p, const uint16_t* pairs, const float* rowsum, const float* coef, float* partials, uint32_t splits, bool wide) {
    const dim3 grid(gemm_q4_dma_blocks(p.m, p.n, p.act_mul != 0, wide), splits);
    return wide ? launch_check([&] { hipLaunchKernelGGL(gemm_q4_dma_kernel<8>, grid, dim3(512), 0, s, p, pairs, rowsum, coef, partials); }, "gemm_q4_dma_wide")
                : launch_check([&] { hipLaunchKernelGGL(gemm_q4_dma_kernel<4>, grid, dim3(256), 0, s, p, pairs, rowsum, coef, partials); }, "gemm_q4_dma");
}

} // namespace k
} // namespace uzu
