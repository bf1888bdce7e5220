// gemm128_epilogue.h -- how a wave's 64 x 64 tile of the large-tile prefill GEMMs (k_gemm128.hip, k_gemm_dma.hip) ends: offset term, epilogue, stores.
#pragma once
#include <type_traits>

#include "device_utils.h"
#include "gemm_convert.h"
#include "kernels.h"
#include "uzu_math.h"

namespace uzu {
namespace k {

// activate_bf16_tab of a gate that holds a bf16 number: SiLU by the hardware's exp2 and reciprocal.  -x times log2 e's leading 15 bits is exact, the rest of the constant joins
// as a factor (its square, dropped, is 0.6 ulp at 80; the exponential, the reciprocal and three roundings 1 or 1/2 each): the quotient is within 8 f32 ulps, and silu_bf16_near has the 64-bit exponential decide where that could change the
// bf16 rounding.  4096 x 28672 x 4096: 1145 -> 1081 us.
__device__ __forceinline__ float gate_act(uint32_t act, float x, const uint64_t* tab) {
    if (act != 0) return activate_bf16_tab(act, x, tab);
    const float e = __builtin_amdgcn_exp2f(x * -0x1.7154p+0f), c = x * (float)(-0x1.d94ae0bf8p-18 * 0x1.62e42fefa39efp-1);
    return silu_bf16_near(x, x * __builtin_amdgcn_rcpf(1.0f + fmaf(e, c, e)), tab);
}

struct GemmTile {
    uint32_t m_w, n_w;        // the wave's first row, first column
    uint32_t n_pair, part;    // gated: first output column of the wave pair, and its 64-column part
    uint32_t ncol[2];         // the lane's column of the weight matrix in each 32-column block (clamped)
    uint32_t wave, wn;        // gated: waves 2 i and 2 i + 1 hold the up and the gate columns of the same outputs
    uint32_t M, Mst, N, H;    // Mst: row bound of every store; H = N / 2
    uint32_t g_lo, g_end, z;  // quant groups of this split, the split
    bool gated, live;
};

// `s_ep`: 9216 bytes per wave that nobody else uses any more; gated: every wave of the workgroup comes here (one workgroup barrier)
template <bool PAIRS>
__device__ __forceinline__ void gemm_tile_finish(const MatmulParams& p, const GemmTile& t, const float* rowsum, const float* coef, float* partials, f32x16_t (&acc_t)[2][2], uint8_t* s_ep, uint64_t* s_exp_tab) {
    const int lane = threadIdx.x & 63, h = lane >> 5, c = lane & 31;
    const uint32_t M = t.M, N = t.N, H = t.H;
    // ---- offset term: acc_t[m, n] += sum_g rowsum[g][m] * coef[g][n] over this split's groups, on the matrix cores in
    // f32 (v_mfma_f32_32x32x2_f32: products and sums exact to f32): lane (c, h) supplies row / column c of group 2 i + h,
    // every load is one coalesced dword per lane.
    if (p.b_kind != UZU_MATMUL_B_SCALE_SYMMETRIC || PAIRS) {
        const uint32_t Mp = (M + 3) & ~3u;
        uint32_t arow[2];
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) arow[mb] = min(t.m_w + mb * 32 + c, Mp - 1);
        // (a producer may have filed 2^PL partial sums per group, rows [g << PL, (g + 1) << PL) of `rowsum`: added here in part order -- more loads in flight per
        // iteration, the same number of iterations and MFMAs; walking the parts as extra iterations cost the long-K down projections more than the pre-pass saved)
        // The loads of eight steps travel together: with the parts' count a branch inside the step they went one round trip after the other (4096 x 14336 x 2048: 289 -> 281 us).
        auto offsets = [&](auto parts) {
            constexpr uint32_t PL = decltype(parts)::value;
#pragma unroll 8
            for (uint32_t g2 = t.g_lo; g2 < t.g_end; g2 += 2) {
                const uint32_t g = min(g2 + h, t.g_end - 1);
                const bool real = g2 + h < t.g_end;
                float av[2], bv[2];
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
                    const float* rp = rowsum + (size_t)(g << PL) * Mp + arow[mb];
                    av[mb] = rp[0];
#pragma unroll
                    for (uint32_t i = 1; i < (1u << PL); ++i) av[mb] += rp[i * (size_t)Mp];
                }
#pragma unroll
                for (int nb = 0; nb < 2; ++nb) {
                    const float v = coef[(size_t)g * N + t.ncol[nb]];
                    bv[nb] = real ? v : 0.f;
                }
#pragma unroll
                for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                    for (int nb = 0; nb < 2; ++nb) acc_t[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[mb], bv[nb], acc_t[mb][nb], 0, 0, 0);
            }
        };
        if (p.rowsum_parts_log2 == 0) offsets(std::integral_constant<uint32_t, 0>()); // (<= 2: host-checked)
        else if (p.rowsum_parts_log2 == 1) offsets(std::integral_constant<uint32_t, 1>());
        else offsets(std::integral_constant<uint32_t, 2>());
    }

    // ---- epilogue (kernel.rs:281-292): lane holds column n, rows (r & 3) + 8 (r >> 2) + 4 h of each block
    uint16_t* d = (uint16_t*)p.d;
    float* d32 = (float*)p.d;
    const bool out_f32 = p.d_dt == UZU_F32;
    const bool via_lds = !partials && !out_f32 && !p.accumulate && !p.has_soft_cap && (t.gated ? H : N) % 8 == 0 && (uintptr_t)p.d % 16 == 0; // gated: host-checked
    if (via_lds) {
        // Common case, branch-free: bf16(ab_scale * acc + bias) goes to a wave-private LDS tile (64 rows x 64 columns,
        // 144-byte pitch; the activation buffers are free after the last barrier) and leaves as 16-byte row segments,
        // 8 lanes per 128-byte row -- instead of 64 two-byte stores per lane.
        uint16_t* s_d = (uint16_t*)s_ep + t.wave * (64 * 72);
        const float ab = p.ab_scale;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            const float bias = p.bias ? bf16_to_f32(((const uint16_t*)p.bias)[t.ncol[nb]]) : 0.0f;
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int r = 0; r < 16; r += 2) { // rows r and r + 1 are consecutive
                    const uint32_t lr = mb * 32 + (r & 3) + 8 * (r >> 2) + 4 * h;
                    const uint32_t pk = pack_bf16(__fadd_rn(__fmul_rn(ab, acc_t[mb][nb][r]), bias), __fadd_rn(__fmul_rn(ab, acc_t[mb][nb][r + 1]), bias)); // two roundings, as the reference
                    s_d[lr * 72 + nb * 32 + c] = (uint16_t)pk;
                    s_d[(lr + 1) * 72 + nb * 32 + c] = (uint16_t)(pk >> 16);
                }
        }
        const int seg = lane & 7, rsub = lane >> 3;
        if (t.gated) {
            // the up tile (wave wm * 2) and the gate tile (wave wm * 2 + 1) hold the same (row, column) positions:
            // out = bf16(up * act(gate)), both operands already rounded to bf16 as the separate kernels would see them; each of the
            // pair's waves combines 32 of the 64 rows; the exp table of SiLU / softplus sits in LDS (a table read from memory per
            // element is a dependent round trip with two waves to hide it)
            if (threadIdx.x < 32) s_exp_tab[threadIdx.x] = kExp2fTab[threadIdx.x];
            __syncthreads();
            const uint16_t* s_u = (const uint16_t*)s_ep + (t.wave & ~1u) * (64 * 72);
            const uint16_t* s_g = s_u + 64 * 72;
#pragma unroll
            for (int pass = 0; pass < 4; ++pass) {
                const uint32_t lr = (t.wn & 1) * 32 + pass * 8 + rsub, m = t.m_w + lr, n = t.n_pair + seg * 8;
                const u32x4_v uv = *(const u32x4_v*)(s_u + lr * 72 + seg * 8), gv = *(const u32x4_v*)(s_g + lr * 72 + seg * 8);
                u32x4_v ov;
                float even = 0.f, part = 0.f; // the row's sum over this lane's 8 ROUNDED outputs (columns past H count as zero)
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const float u0 = bits_to_f32(uv[w] << 16), u1 = bits_to_f32(uv[w] & 0xFFFF0000u);
                    const float g0 = bits_to_f32(gv[w] << 16), g1 = bits_to_f32(gv[w] & 0xFFFF0000u);
                    ov[w] = pack_bf16(u0 * gate_act(p.act_type, g0, s_exp_tab), u1 * gate_act(p.act_type, g1, s_exp_tab));
                    (p.d_pairs ? even : part) += bits_to_f32(ov[w] << 16); // (rows in pair order: the pre-pass's order of summation, which they would have been left to)
                    part += bits_to_f32(ov[w] & 0xFFFF0000u);
                }
                if (p.d_pairs) part = even + part;
                if (m < t.Mst && n < H) *(u32x4_v*)(d + (size_t)m * H + n) = p.d_pairs ? permute_pairs(ov) : ov;
                if (p.gated_rowsum_out) { // the 8 lanes of a row segment group are neighbours: three butterfly steps, lane seg 0 files the 64-column sum
                    if (n >= H) part = 0.f;
                    part += __shfl_xor(part, 1);
                    part += __shfl_xor(part, 2);
                    part += __shfl_xor(part, 4);
                    const uint32_t Mp = (M + 3) & ~3u;
                    if (seg == 0 && t.live && m < Mp) p.gated_rowsum_out[(size_t)t.part * Mp + m] = m < M ? part : 0.f;
                }
            }
        } else {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // wave-private region: no workgroup barrier needed
#pragma unroll
            for (int pass = 0; pass < 8; ++pass) {
                const uint32_t lr = pass * 8 + rsub, m = t.m_w + lr, n = t.n_w + seg * 8;
                const u32x4_v v = *(const u32x4_v*)(s_d + lr * 72 + seg * 8);
                if (m < t.Mst && n < N) *(u32x4_v*)(d + (size_t)m * N + n) = v;
            }
        }
    } else if (partials) { // split-K: raw f32 partial tile (32 lanes = one 128-byte row segment per store)
        float* pz = partials + (size_t)t.z * M * N;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            const uint32_t n = t.n_w + nb * 32 + c;
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t m = t.m_w + mb * 32 + (r & 3) + 8 * (r >> 2) + 4 * h;
                    if (m < t.Mst && n < N) pz[(size_t)m * N + n] = acc_t[mb][nb][r];
                }
        }
    } else {
#pragma unroll 1
        for (int nb = 0; nb < 2; ++nb) {
            const uint32_t n = t.n_w + nb * 32 + c;
            const float bias = (p.bias && n < N) ? bf16_to_f32(((const uint16_t*)p.bias)[n]) : 0.0f;
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t m = t.m_w + mb * 32 + (r & 3) + 8 * (r >> 2) + 4 * h;
                    if (m >= t.Mst || n >= N) continue;
                    const size_t idx = (size_t)m * N + n;
                    const float acc = nb ? acc_t[mb][1][r] : acc_t[mb][0][r];
                    float value = p.ab_scale * acc;
                    if (p.accumulate) value += out_f32 ? d32[idx] : bf16_to_f32(d[idx]);
                    if (p.bias) value += bias;
                    if (p.has_soft_cap) value = p.soft_cap * tanhf(value / p.soft_cap);
                    if (out_f32) d32[idx] = value;
                    else d[idx] = f32_to_bf16(value);
                }
        }
    }
}

} // namespace k
} // namespace uzu
