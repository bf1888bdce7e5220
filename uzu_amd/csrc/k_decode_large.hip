// k_decode_large.hip -- the decode GEMV of large matrices (bandwidth regime): gemv_dec's arithmetic (gemv_core.h, bit for bit) as a stream.
//
// gemv_dec (k_decode.hip) holds the activation row in registers, two items of weights in flight a wave and as many workgroups as fit, each with the Normalization in front: 25 MB of a
// qkv projection took two rounds of workgroups, and a row too long for registers was read again from the L2 for every row of the matrix.  Here
//   * a workgroup of eight waves per CU, a row (or up / gate pair) of the matrix a wave and round;
//   * the activation row lies in LDS as f32, once per workgroup, with the sums of its steps of 32;
//   * a wave's share is one sequence of items -- a step of 2048 codes, their scales and offsets -- through D slots of registers: D items are on their way from before the Normalization to
//     the end, across the borders of rows.
// How much is on its way matters both ways.  Nothing but the loads (2048 waves, a row each): 58.7 MB 10.1 us and 525 MB 76 us (6.9 TB/s) with 8 MB in flight, 12.2 and 92 with 32 MB; hence
// the small D, and hence no load that nobody wants (a row past the end lies past its buffer's end and is not fetched).
// Bound by the memory's rate and, below 30 MB or so, by the launch and the Normalization.  Us, Llama-3-8B, gemv_dec -> here: qkv (25 MB, Normalization) 11.9 -> 9.1, out (17 MB) 7.2 -> 5.5,
// up (117 MB, Normalization, GatedActMul) 25.9 -> 23.3, down (59 MB) 17.6 -> 12.1, read-out (525 MB) 101 -> 84.
#include <stdlib.h>

#include <algorithm>

#include "decode_epilogue.h"
#include "device_utils.h"
#include "gemv_core.h"
#include "kernels.h"
#include "kernels_decode.h"

namespace uzu {
namespace k {

namespace {
constexpr int NWL = 8, NTL = 64 * NWL;
constexpr int kSlotFloats = 36; // a step's 32 numbers and 16 bytes: reads of 16 neighbouring steps fall on different banks

template <int NPHYS> struct Item {
    gc_u32x4 a[NPHYS], b[NPHYS];
    uint32_t s[NPHYS], o[NPHYS]; // (32-bit: held across the loop)
};
// A lane's numbers are the 32 codes of one step (gemv_dec's mapping), but its loads are 16 bytes of either KB of the row's 2 KB, so that an instruction takes whole lines (at 32 bytes
// a lane every line is asked for twice: 58.7 MB 11.3 us against 10.1).  Lane 2 m has the first halves and lane 2 m + 1 the second halves of steps m and 32 + m: neighbours swap, and lane l
// owns step l / 2 + 32 (l & 1).
__device__ __forceinline__ void own_step(Codes8& c, const gc_u32x4& a, const gc_u32x4& b, bool odd) {
    uint32_t first[4], second[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const uint32_t u = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(odd ? a[w] : b[w]), 0xB1, 0xF, 0xF, true); // the neighbour's
        first[w] = odd ? u : a[w], second[w] = odd ? b[w] : u;
    }
    c.a = make_uint4(first[0], first[1], first[2], first[3]), c.b = make_uint4(second[0], second[1], second[2], second[3]);
}
__device__ __forceinline__ uint32_t step_place(uint32_t c) { return (c & ~63u) | ((c & 31u) << 1) | ((c >> 5) & 1u); } // of step c in LDS: the lane that owns it
__device__ __forceinline__ void load_slot(const float* xs, uint32_t place, float (&x)[32]) {
    const f32x4_v* src = (const f32x4_v*)(xs + (size_t)place * kSlotFloats);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const f32x4_v t = src[i];
        x[4 * i] = t.x, x[4 * i + 1] = t.y, x[4 * i + 2] = t.z, x[4 * i + 3] = t.w;
    }
}

// PRO: the Normalization of the row (k <= 8192) in front; ACT: rows come in pairs [up | gate] and leave as GatedActMul
template <int D, bool PRO, bool ACT>
__global__ void __launch_bounds__(NTL, 2) gemv_large_kernel(DecGemvParams p) {
    constexpr int NPHYS = ACT ? 2 : 1;
    extern __shared__ __attribute__((aligned(16))) float smem[];
    __shared__ float red[4];
    __shared__ uint64_t s_exp_tab[ACT ? 32 : 1];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t K = p.k, C = K / 32, P = C / 64, gshift = 31 - __builtin_clz(p.group_size), G = K >> gshift;
    float* const xs = smem;                             // [C][36]
    float* const xsum = smem + (size_t)C * kSlotFloats; // [C]
    const uint32_t n0 = ACT ? p.n[0] / 2 : p.n[0], rows = n0 + (ACT ? 0u : p.n[1]), W = gridDim.x * NWL;
    const uint32_t b0 = blockIdx.x * NWL + wave;

    // ---- the stream's loads, unconditional (a branch around them would make every wait a wait for all of them): a row past the matrix' end lies past its buffer's end
    auto rsrc = [&](const void* base, uint64_t bytes) { return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)(uint32_t)std::min<uint64_t>(bytes, 0xFFFFFFFFull), 0x00027000); };
    const auto w_rs0 = rsrc(p.w[0], (uint64_t)p.n[0] * K), w_rs1 = rsrc(p.w[1], (uint64_t)p.n[1] * K);
    const auto s_rs0 = rsrc(p.scales[0], (uint64_t)p.n[0] * G * 2), s_rs1 = rsrc(p.scales[1], (uint64_t)p.n[1] * G * 2), o_rs0 = rsrc(p.biases[0], (uint64_t)p.n[0] * G * 2), o_rs1 = rsrc(p.biases[1], (uint64_t)p.n[1] * G * 2);
    uint32_t lb = b0, lj = 0;
    const uint32_t step = (lane >> 1) + (lane & 1) * 32; // of 64: the lane's
    const bool odd = lane & 1;
    auto load = [&](Item<NPHYS>& it) {
        const bool second = __builtin_amdgcn_readfirstlane(!ACT && lb >= n0 ? 1 : 0);
        const uint32_t first = second ? lb - n0 : lb, at0 = lj * 2048 + lane * 16, grp = ((lj * 64 + step) * 32) >> gshift;
        const bool in = lb < rows;
        const auto w_rs = second ? w_rs1 : w_rs0;
        const auto s_rs = second ? s_rs1 : s_rs0;
        const auto o_rs = second ? o_rs1 : o_rs0;
#pragma unroll
        for (int h = 0; h < NPHYS; ++h) {
            const uint32_t row = first + (h ? n0 : 0u), at = in ? row * K + at0 : 0xFFFFF000u, gi = in ? (row * G + grp) * 2 : 0xFFFFF000u;
            it.a[h] = __builtin_amdgcn_raw_buffer_load_b128(w_rs, at, 0, 2), it.b[h] = __builtin_amdgcn_raw_buffer_load_b128(w_rs, at + 1024, 0, 2); // (nt)
            it.s[h] = __builtin_amdgcn_raw_buffer_load_b16(s_rs, gi, 0, 0), it.o[h] = __builtin_amdgcn_raw_buffer_load_b16(o_rs, gi, 0, 0);
        }
        const bool last = lj + 1 == P;
        lj = last ? 0 : lj + 1;
        lb = last ? lb + W : lb;
    };
    Item<NPHYS> it[D];

    // ---- the activation row: requested in front of the weights (loads return in order)
    constexpr int NPRE = PRO ? 8 : 1;
    u32x2_v x_pre[NPRE], s_pre[NPRE];
    f32x4_v n_pre[NPRE];
    constexpr int XST = PRO ? 1 : 2; // steps staged a thread (k <= 32768)
    gc_raw4 x_raw[XST][4];
    const uint32_t E = K / 256; // Normalization: thread t of the first 256 owns elements [t E, t E + E) (normalization_kernel's mapping)
    if constexpr (PRO) {
        if (wave < 4)
#pragma unroll
            for (int qi = 0; qi < NPRE; ++qi) {
                const uint32_t q = (uint32_t)qi * 4 < E ? (uint32_t)qi * 4 : E - 4, e = tid * E + q;
                x_pre[qi] = *(const u32x2_v*)(p.x + e);
                s_pre[qi] = *(const u32x2_v*)((p.residual_add ? p.shortcut_in : p.x) + e);
                n_pre[qi] = *(const f32x4_v*)(p.norm_scales ? p.norm_scales + e : (const float*)p.x);
            }
    } else {
#pragma unroll
        for (int q = 0; q < XST; ++q) {
            const gc_raw4* src = (const gc_raw4*)(p.x + (size_t)min(tid + NTL * q, C - 1) * 32);
#pragma unroll
            for (int w = 0; w < 4; ++w) x_raw[q][w] = src[w];
        }
    }
    uint64_t exp_entry = 0;
    if (ACT) exp_entry = kExp2fTab[tid & 31];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < D; ++u) load(it[u]);
    __builtin_amdgcn_sched_barrier(0);

    if (ACT && tid < 32) s_exp_tab[tid] = exp_entry;
    if constexpr (PRO) { // Normalization (normalization.rs:56-125), order of normalization_kernel
        float ss = 0.f;
        if (wave < 4) {
#pragma unroll
            for (int qi = 0; qi < NPRE; ++qi) {
                const uint32_t q = (uint32_t)qi * 4, e = tid * E + q;
                if (q >= E) break;
                float v[4] = {bits_to_f32(x_pre[qi].x << 16), bits_to_f32(x_pre[qi].x & 0xFFFF0000u), bits_to_f32(x_pre[qi].y << 16), bits_to_f32(x_pre[qi].y & 0xFFFF0000u)};
                if (p.residual_add) {
                    const float sc[4] = {bits_to_f32(s_pre[qi].x << 16), bits_to_f32(s_pre[qi].x & 0xFFFF0000u), bits_to_f32(s_pre[qi].y << 16), bits_to_f32(s_pre[qi].y & 0xFFFF0000u)};
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = round_bf16(v[i] + sc[i]);
                }
                if (p.shortcut_out && blockIdx.x == 0) {
                    u32x2_v o;
                    o.x = (f32_to_bits(v[0]) >> 16) | (f32_to_bits(v[1]) & 0xFFFF0000u), o.y = (f32_to_bits(v[2]) >> 16) | (f32_to_bits(v[3]) & 0xFFFF0000u);
                    *(u32x2_v*)(p.shortcut_out + e) = o;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) ss = fmaf(v[i], v[i], ss);
                *(f32x4_v*)(xs + (size_t)step_place(e / 32) * kSlotFloats + e % 32) = f32x4_v{v[0], v[1], v[2], v[3]};
            }
            ss = wave_sum(ss);
            if (lane == 0) red[wave] = ss;
        }
        lds_barrier();
        if (wave < 4) {
            const float rms_inv = 1.0f / sqrtf((((red[0] + red[1]) + red[2]) + red[3]) / (float)K + p.norm_eps);
#pragma unroll
            for (int qi = 0; qi < NPRE; ++qi) {
                const uint32_t q = (uint32_t)qi * 4, e = tid * E + q;
                if (q >= E) break;
                float* slot = xs + (size_t)step_place(e / 32) * kSlotFloats + e % 32; // own elements: no barrier needed
                f32x4_v v = *(const f32x4_v*)slot;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float normalized = v[i] * rms_inv, scl = n_pre[qi][i];
                    if (!p.norm_scales) v[i] = round_bf16(normalized);
                    else if (p.norm_full_layer) v[i] = round_bf16(normalized * (scl + p.norm_offset));
                    else v[i] = round_bf16(round_bf16(normalized) * round_bf16(scl + p.norm_offset));
                }
                *(f32x4_v*)slot = v;
                if (p.normed_out && blockIdx.x == 0) {
                    u32x2_v o;
                    o.x = (f32_to_bits(v[0]) >> 16) | (f32_to_bits(v[1]) & 0xFFFF0000u), o.y = (f32_to_bits(v[2]) >> 16) | (f32_to_bits(v[3]) & 0xFFFF0000u);
                    *(u32x2_v*)(p.normed_out + e) = o;
                }
            }
        }
        lds_barrier();
    } else {
#pragma unroll
        for (int q = 0; q < XST; ++q) {
            const uint32_t c = tid + NTL * q;
            if (c >= C) break;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const gc_raw4 u = x_raw[q][w];
                float* to = xs + (size_t)step_place(c) * kSlotFloats + 8 * w;
                *(f32x4_v*)to = f32x4_v{bits_to_f32(u.x << 16), bits_to_f32(u.x & 0xFFFF0000u), bits_to_f32(u.y << 16), bits_to_f32(u.y & 0xFFFF0000u)};
                *(f32x4_v*)(to + 4) = f32x4_v{bits_to_f32(u.z << 16), bits_to_f32(u.z & 0xFFFF0000u), bits_to_f32(u.w << 16), bits_to_f32(u.w & 0xFFFF0000u)};
            }
        }
        lds_barrier();
    }
    for (uint32_t c = tid; c < C; c += NTL) {
        float x[32];
        load_slot(xs, c, x);
        xsum[c] = sum32(x);
    }
    lds_barrier();

    float best_v = -INFINITY, keep_up = 0.f, keep_gate = 0.f;
    uint32_t best_i = 0xFFFFFFFFu, keep_row = 0xFFFFFFFFu, kept = 0;
    auto act_flush = [&]() { // a finished pair parks in a lane: the activation runs once for 64 of them (gated_act_mul/mod.rs:5-12)
        if (keep_row != 0xFFFFFFFFu) p.out[0][keep_row] = f32_to_bf16(round_bf16(keep_up * act_bf16(p.act_type, keep_gate, s_exp_tab)));
        keep_row = 0xFFFFFFFFu, kept = 0;
    };
    uint32_t cb = b0, cj = 0;
    float acc[NPHYS];
#pragma unroll
    for (int h = 0; h < NPHYS; ++h) acc[h] = 0.f;
    const int home = (lane < 32 ? 2 * lane : 2 * (lane - 32) + 1) * 4; // the lane that owns step `lane`: the row's sum in the order of the steps
    while (cb < rows) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
            if (cb < rows) {
                const uint32_t place = cj * 64 + lane;
                const float xsm = xsum[place];
                float x[32];
                load_slot(xs, place, x);
#pragma unroll
                for (int h = 0; h < NPHYS; ++h) {
                    Codes8 codes;
                    own_step(codes, it[u].a[h], it[u].b[h], odd);
                    acc[h] = fmaf(bits_to_f32(it[u].s[h] << 16), dot32(codes, x), fmaf(bits_to_f32(it[u].o[h] << 16), xsm, acc[h]));
                    __builtin_amdgcn_sched_barrier(0); // one row at a time: interleaved, the converted codes of both would be live
                }
                if (++cj == P) {
                    const uint32_t mat = __builtin_amdgcn_readfirstlane(!ACT && cb >= n0 ? 1 : 0), row = mat ? cb - n0 : cb;
                    float v[NPHYS];
#pragma unroll
                    for (int h = 0; h < NPHYS; ++h) v[h] = wave_sum(__builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(home, __builtin_bit_cast(int, acc[h])))), acc[h] = 0.f;
                    if constexpr (ACT) { // MatmulKernel epilogue with ab_scale = 1 (kernel.rs:281-292), rounded to bf16
                        float up = v[0], gate = v[NPHYS - 1];
                        if (p.out_bias[0]) up += bf16_to_f32(p.out_bias[0][row]), gate += bf16_to_f32(p.out_bias[0][row + n0]);
                        if (lane == kept) keep_up = round_bf16(up), keep_gate = round_bf16(gate), keep_row = row;
                        if (++kept == 64) act_flush();
                    } else if (lane == 0) {
                        float value = v[0];
                        if (p.out_bias[mat]) value += bf16_to_f32(p.out_bias[mat][row]);
                        const uint16_t ob = f32_to_bf16(value);
                        if (p.out_f32) p.out_f32[row] = value;
                        else p.out[mat][row] = ob;
                        const float lv = bf16_to_f32(ob);
                        if (p.part_val && (lv > best_v || (lv == best_v && row < best_i))) best_v = lv, best_i = row;
                    }
                    cj = 0, cb += W;
                }
            }
            load(it[u]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if constexpr (ACT) act_flush();
    else if (p.part_val) { // UnifiedSampling (greedy) pass 1: one (value, index) partial per workgroup; lane 0 of a wave holds its best
        __shared__ float sv[NWL];
        __shared__ uint32_t si[NWL];
        if (lane == 0) sv[wave] = best_v, si[wave] = best_i;
        __syncthreads();
        if (tid == 0) {
            for (int w = 1; w < NWL; ++w)
                if (sv[w] > best_v || (sv[w] == best_v && si[w] < best_i)) best_v = sv[w], best_i = si[w];
            p.part_val[blockIdx.x] = best_v, p.part_idx[blockIdx.x] = best_i;
        }
    }
}

size_t large_lds(uint32_t k) { return (size_t)(k / 32) * (kSlotFloats + 1) * 4; }
template <int D, bool PRO, bool ACT> uzu_status launch_large(hipStream_t s, const DecGemvParams& p, uint32_t grid) {
    const size_t lds = large_lds(p.k);
    static LdsLimit lim;
    UZU_REQUIRE(raise_lds_limit(lim, (const void*)gemv_large_kernel<D, PRO, ACT>, lds), "gemv_large: %zu bytes of LDS are not available", lds);
    return launch_check([&] { hipLaunchKernelGGL((gemv_large_kernel<D, PRO, ACT>), dim3(grid), dim3(NTL), lds, s, p); }, "gemv_large");
}
template <int D, bool ACT> uzu_status launch_large_p(hipStream_t s, const DecGemvParams& p, uint32_t grid) {
    return p.norm_scales || p.norm_plain ? launch_large<D, true, ACT>(s, p, grid) : launch_large<D, false, ACT>(s, p, grid);
}
} // namespace

// int8 with bf16 scales and offsets, whole steps of a wave, from 8 MB on (below, a CU's share is over before the row is staged).  int4 is not better off: its conversion wants the sixteen
// waves of gemv_dec (Llama-3-8B's up, down and read-out 16.3 / 9.0 / 50.9 us there, 17.3 / 9.5 / 68.5 as a stream).
// Gated rows: gemv_dec holds four pairs a CU at once, of K = 2048 twelve, and is the faster one up to there (up / gate, us, gemv_dec and here: 2048 x 4096 6.7 / 8.3, 2144 x 4096 9.0 / 8.4, 2048 x 8192
// 12.7 / 13.0, 2560 x 8192 17.4 / 13.4, 6144 x 2048 7.7 / 8.0, 6400 x 2048 9.3 / 8.1).
bool gemv_large_wanted(const DecGemvParams& p, int num_cus) {
    const bool normed = p.norm_scales || p.norm_plain;
    if (p.bits != 8 || p.b_kind != UZU_MATMUL_B_SCALE_BIAS || p.k % 2048 || p.k > 32768 || p.group_size < 32 || (p.group_size & (p.group_size - 1)) || p.k % p.group_size || (normed && p.k > 8192)) return false;
    if (p.conv_w || p.dg_o || p.x_rht_bits || p.in_rht_bits || p.ep_out_bits || (p.act_mul && (p.n[1] || p.part_val || p.out_f32))) return false;
    if (p.act_mul && p.n[0] / 2 <= (p.k == 2048 ? 12u : 4u) * (uint32_t)num_cus) return false;
    return (uint64_t)std::max(p.n[0], p.n[1]) * p.k < 0xFFFFF000ull && ((uint64_t)p.n[0] + p.n[1]) * p.k >= (8ull << 20);
}
uzu_status gemv_large(hipStream_t s, const DecGemvParams& p, int num_cus, uint32_t* grid_out) {
    uint32_t grid = (uint32_t)num_cus;
    if (p.part_val && p.part_capacity && grid > p.part_capacity) grid = p.part_capacity;
    const uint32_t rows = (p.act_mul ? p.n[0] / 2 : p.n[0]) + p.n[1];
    grid = std::min(grid, (rows + NWL - 1) / NWL);
    if (grid_out) *grid_out = grid;
    if (p.act_mul) return launch_large_p<2, true>(s, p, grid);
    // 8 MB of items on their way; 12 where the stream is long (2 and 3 items a wave, us: 16.8 MB 5.5 / 5.9, 25 MB 9.1 / 9.5, 58.7 MB 12.1 / 12.3, 525 MB 87.2 / 84.1)
    return (uint64_t)rows * p.k >= (128ull << 20) ? launch_large_p<3, false>(s, p, grid) : launch_large_p<2, false>(s, p, grid);
}

} // namespace k
} // namespace uzu
