// k_linear_mfma.hip -- the full-precision linear of the f32-stream designs on the bf16 matrix cores (kernels_stream32.h: linear_f32).  Two forms: operands staged through
// registers (below), and operand rows converted once and brought by LDS DMA (linear_dma_kernel: larger products, products cut along k, true f32 products as three bf16 parts).
//
//   Y[r, n] = act(sum_k bf16(X[r, k]) * W[n, k] + bias[n]) + residual[r, n]       X f32 rows, W bf16 [n, k], f32 accumulation, f32 out
//
// v_mfma_f32_32x32x16_bf16; a workgroup of four waves (2 x 2) owns a (64 MB) x (64 NB) tile, a wave MB x NB blocks of 32 x 32.  A k-step is 64 deep: the
// activation rows are rounded to bf16 on their way into LDS (what a bf16 activation buffer would have held -- the round trip through HBM is saved instead of
// the conversion), the weight rows are copied; both tiles use a 144-byte row pitch, so the 16-byte operand reads of the 64 lanes fall on distinct banks.
// The next k-step's global loads are issued before the MFMAs of the current one and stored behind them (one LDS buffer, two barriers per k-step).
// An MFMA lane holds column n = lane % 32 of a block and rows (i & 3) + 8 (i >> 2) + 4 (lane / 32): a row's 32 columns leave as one 128-byte segment.
// grid.z batches independent products of one shape (the per-head products of the latent attention).
#include <algorithm>

#include "device_utils.h"
#include "gemm_convert.h"
#include "gemm_tile_order.h"
#include "kernels.h"
#include "kernels_stream32.h"
#include "stream32_epilogue.h"

namespace uzu {
namespace k {

namespace {

constexpr int LK = 64;       // k-step
constexpr int PITCH = 144;   // bytes per staged row: 64 bf16 + 16 bytes of pad

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) { return (uint32_t)f32_to_bf16(a) | ((uint32_t)f32_to_bf16(b) << 16); }

template <int MB, int NB, bool GROUPED, int KIND> // KIND: EpilogueKind; GROUPED: per-product row buckets (row_offsets) and gathered operand rows (row_map); the plain form carries neither
__global__ void __launch_bounds__(256, MB * NB == 4 && KIND != kEpilogueFull ? 3 : 1) linear_mfma_kernel(LinearF32Params p) {
    constexpr int BM = 64 * MB, BN = 64 * NB;
    constexpr int A_PASSES = BM / 16; // 16 threads cover a row's 64 k (one float4 each), 16 rows per pass
    constexpr int B_PASSES = BN / 32; // 8 threads cover a row's 64 k (one 16-byte vector each), 32 rows per pass
    __shared__ __attribute__((aligned(16))) uint8_t s_a[BM * PITCH];
    __shared__ __attribute__((aligned(16))) uint8_t s_b[BN * PITCH];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave >> 1, wn = wave & 1, l32 = lane & 31, half = lane >> 5;
    const uint32_t z = blockIdx.z;
    const float* x = p.x + z * p.x_batch;
    const uint16_t* w = p.w + z * p.w_batch;
    uint32_t r_lo = 0, r_hi = p.rows;
    if (GROUPED) { // a grouped launch: this product's bucket of rows (workgroup-uniform: the exit comes before any barrier)
        r_lo = p.row_offsets[z], r_hi = p.row_offsets[z + 1];
        x = p.x;
    }
    const uint32_t m0 = r_lo + blockIdx.y * BM, n0 = blockIdx.x * BN;
    if (m0 >= r_hi) return;

    f32x16_t acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    f32x4_v a_reg[A_PASSES];
    u32x4_v b_reg[B_PASSES];
    const uint32_t a_row = tid >> 4, a_k = (tid & 15) * 4;
    const uint32_t b_row = tid >> 3, b_k = (tid & 7) * 8;
    // GROUPED: where this thread's rows start, once (element offsets; the gather's indices must not be read again in every k-step): a row or column outside the product
    // is read from inside it and its sums are not stored
    uint32_t a_at[A_PASSES], b_at[B_PASSES];
    if (GROUPED) {
#pragma unroll
        for (int i = 0; i < A_PASSES; ++i) {
            const uint32_t r = m0 + a_row + i * 16, in = r < r_hi ? r : r_hi - 1;
            a_at[i] = (p.row_map ? p.row_map[in] : in) * p.ldx + a_k;
        }
#pragma unroll
        for (int i = 0; i < B_PASSES; ++i) {
            const uint32_t n = n0 + b_row + i * 32;
            b_at[i] = (n < p.n ? n : p.n - 1) * p.k + b_k;
        }
    }
    auto load = [&](uint32_t k0) {
        if (GROUPED) {
            const bool a_ok = k0 + a_k < p.k, b_ok = k0 + b_k < p.k; // (the last k-step)
#pragma unroll
            for (int i = 0; i < A_PASSES; ++i) {
                const f32x4_v v = *(const f32x4_v*)(x + (a_ok ? a_at[i] + k0 : 0u));
                a_reg[i] = a_ok ? v : f32x4_v{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int i = 0; i < B_PASSES; ++i) {
                const u32x4_v v = *(const u32x4_v*)(w + (b_ok ? b_at[i] + k0 : 0u));
                b_reg[i] = b_ok ? v : u32x4_v{0u, 0u, 0u, 0u};
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < A_PASSES; ++i) {
            const uint32_t r = m0 + a_row + i * 16, kk = k0 + a_k;
            const bool ok = r < r_hi && kk < p.k;
            const float* src = x + (size_t)(ok ? r : 0) * p.ldx + (ok ? kk : 0);
            const f32x4_v v = *(const f32x4_v*)src;
            a_reg[i] = ok ? v : f32x4_v{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < B_PASSES; ++i) {
            const uint32_t n = n0 + b_row + i * 32, kk = k0 + b_k;
            const bool ok = n < p.n && kk < p.k;
            const uint16_t* src = w + (size_t)(ok ? n : 0) * p.k + (ok ? kk : 0);
            const u32x4_v v = *(const u32x4_v*)src;
            b_reg[i] = ok ? v : u32x4_v{0u, 0u, 0u, 0u};
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int i = 0; i < A_PASSES; ++i) {
            const uint32_t row = a_row + i * 16;
            u32x2_v o;
            o.x = pack_bf16(a_reg[i].x, a_reg[i].y), o.y = pack_bf16(a_reg[i].z, a_reg[i].w);
            *(u32x2_v*)(s_a + row * PITCH + a_k * 2) = o;
        }
#pragma unroll
        for (int i = 0; i < B_PASSES; ++i) {
            const uint32_t row = b_row + i * 32;
            *(u32x4_v*)(s_b + row * PITCH + b_k * 2) = b_reg[i];
        }
    };

    load(0);
    for (uint32_t k0 = 0; k0 < p.k; k0 += LK) {
        __syncthreads(); // the MFMAs of the step before have read the tiles
        stage();
        __syncthreads();
        if (k0 + LK < p.k) load(k0 + LK);
#pragma unroll
        for (int s = 0; s < LK / 16; ++s) {
            u32x4_t af[MB], bfr[NB];
#pragma unroll
            for (int i = 0; i < MB; ++i) af[i] = *(const u32x4_t*)(s_a + ((wm * MB + i) * 32 + l32) * PITCH + (s * 16 + half * 8) * 2);
#pragma unroll
            for (int j = 0; j < NB; ++j) bfr[j] = *(const u32x4_t*)(s_b + ((wn * NB + j) * 32 + l32) * PITCH + (s * 16 + half * 8) * 2);
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, af[i]), __builtin_bit_cast(bf16x8_t, bfr[j]), acc[i][j], 0, 0, 0);
        }
    }

    float* y = GROUPED ? p.y : p.y + z * p.y_batch;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const uint32_t n = n0 + (wn * NB + j) * 32 + l32;
        if (n >= p.n) continue;
        const float bias = p.bias ? bf16_to_f32(p.bias[n]) : 0.0f;
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            const uint32_t row0 = m0 + (wm * MB + i) * 32 + 4 * half;
            float res[16]; // (the residual may be y itself: a block's rows are read before any of them is stored)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t row = row0 + (r & 3) + 8 * (r >> 2);
                res[r] = p.residual && row < r_hi ? p.residual[(size_t)row * p.ldr + n] : 0.0f;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t row = row0 + (r & 3) + 8 * (r >> 2);
                if (row >= r_hi) continue;
                const float v = linear_value<KIND>(acc[i][j][r], bias, p, row, z, n);
                y[(size_t)row * p.ldy + n] = p.residual ? v + res[r] : v;
            }
        }
    }
}


// ---- prompt-sized products: both operands as bf16 rows in memory, fetched straight into LDS
// The activations are rounded to bf16 once, in front (linear_bf16_rows, or the producing kernel), instead of by every column of tiles: the kernel above spends its
// k-step on that conversion and on the operands' way through registers (2048 x 7712 x 2048: 158 us, 409 TFLOP/s), with one buffer and two barriers per k-step.
// Here a workgroup of WM x WN waves, a wave 32 MB x 64 outputs, takes its 64-deep k-steps by global_load_lds_dwordx4 (1 KB a wave-instruction, no registers).
// A staged row is 64 k = 128 bytes = eight 16-byte chunks; chunk c of row r lies in slot c ^ (r / 2 & 7) -- the lane picks the chunk it fetches, the DMA stores lane by
// lane -- so the sixteen rows that a quarter-wave reads at one k fall on the sixteen different 16-byte slots of two rows.
// What bounds it is the wait for a k-step's operands, so the forms differ in who covers it (measured, us, conversion included):
//   * 128-row tiles, ONE buffer, 32 KB: four workgroups per CU cover each other.  Best from two tiles a CU on: 2048 x 16384 x 2048 183 (two buffers 211),
//     eight buckets of 4096 rows x 4096 x 2048 105 (111), x 2048 59 (67);
//   * 128-row tiles, two buffers, two workgroups per CU, the next step on its way during a step: 513 x 8192 x 2048 45 (one buffer 52);
//   * up to a 128-row tile a CU: eight waves on it (eight_wave_splits), or 64-row tiles of four waves, two buffers, three workgroups per CU.
// 256 columns or rows a workgroup, eight waves of 64 x 64 or 128 x 64, were slower from two tiles a CU on, too (2048 x 7712 x 2048 97, 94 and 81 us against 82; eight buckets of 512 rows
// x 4096 x 2048 122 .. 136 against 108), as were 32-deep steps.
constexpr int DN = 128;

// PIECES KB-pieces from base + v[i] (16 bytes a lane) to dst + 1024 i + 16 lane
template <int PIECES> __device__ __forceinline__ void dma16(const void* base, const uint32_t (&v)[PIECES], uint32_t dst) {
    uint32_t keep;
    if constexpr (PIECES == 2)
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
                     "global_load_lds_dwordx4 %3, %1\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
                     "global_load_lds_dwordx4 %4, %1\n\ts_mov_b32 m0, %0"
                     : "=&s"(keep) : "s"(base), "s"(dst), "v"(v[0]), "v"(v[1]) : "memory", "scc");
    else {
        static_assert(PIECES == 4, "two or four pieces");
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
                     "global_load_lds_dwordx4 %3, %1\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
                     "global_load_lds_dwordx4 %4, %1\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
                     "global_load_lds_dwordx4 %5, %1\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
                     "global_load_lds_dwordx4 %6, %1\n\ts_mov_b32 m0, %0"
                     : "=&s"(keep) : "s"(base), "s"(dst), "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]) : "memory", "scc");
    }
}

// f32 products on the same matrix cores: an f32 number is three bf16 numbers, x = hi + mid + lo exactly (8 + 8 + 8 significant bits, each part the truncation of what the
// parts before it leave), weights are bf16 already, and a product of two bf16 numbers is exact in f32: the sum over 3 k products, the small parts first, is a sum of the
// f32 products' own bits with f32 accumulation.  Three bf16 products are five times the rate of the f32 matrix instructions.  The small parts are stored 2^7 and 2^14 times
// as large, no part larger than x, and the running sum is scaled back at a part's end: bf16 ends at 2^-133, and unscaled parts lose bits of every x below 2^-110 (here
// below 2^-124).  Infinities and NaNs stay in hi.
constexpr float kPartDown = 1.0f / 128.0f;
__device__ __forceinline__ void split_bf16(float x, uint16_t& hi, uint16_t& mid, uint16_t& lo) {
    const uint32_t u = f32_to_bits(x);
    const bool finite = (u & 0x7F800000u) != 0x7F800000u;
    const float h = bits_to_f32(u & 0xFFFF0000u), r = (x - h) * 128.0f, m = bits_to_f32(f32_to_bits(r) & 0xFFFF0000u);
    hi = finite ? (uint16_t)(u >> 16) : f32_to_bf16(x);
    mid = finite ? (uint16_t)(f32_to_bits(m) >> 16) : (uint16_t)0;
    lo = finite ? (uint16_t)(f32_to_bits((r - m) * 128.0f) >> 16) : (uint16_t)0;
}
// A part that is zero times an infinite weight is a NaN where the f32 product is an infinity (the parts have x's sign, so nothing else can go wrong): a sum that came out as NaN
// is made again from the f32 numbers themselves, one after the other.
__device__ __forceinline__ float split_dot(const uint16_t* xrow, const uint16_t* wrow, uint32_t k) {
    float sum = 0.0f;
#pragma unroll 1
    for (uint32_t c = 0; c < k; ++c)
        sum = fmaf(bf16_to_f32(xrow[2 * k + c]) + (bf16_to_f32(xrow[k + c]) * kPartDown + bf16_to_f32(xrow[c]) * (kPartDown * kPartDown)), bf16_to_f32(wrow[c]), sum);
    return sum;
}
// acc[r] = the sum of row row0 + (r & 3) + 8 (r >> 2) and weight row wrow
__device__ __forceinline__ void split_repair(f32x16_t& acc, const uint16_t* xb, uint32_t k, const uint32_t* row_map, uint32_t row0, uint32_t row_end, const uint16_t* wrow) {
    float all = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) all = fmaxf(all, acc[r] != acc[r] ? 1.0f : 0.0f);
    if (!__builtin_expect(__ballot(all != 0.0f) != 0, 0)) return;
    float sums[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) sums[r] = acc[r];
#pragma unroll 1
    for (uint32_t r = 0; r < 16; ++r) {
        const uint32_t row = row0 + (r & 3) + 8 * (r >> 2);
        if (row < row_end && sums[r] != sums[r]) sums[r] = split_dot(xb + (size_t)(row_map ? row_map[row] : row) * 3 * k, wrow, k);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = sums[r];
}

constexpr int kEpilogueGated = 16; // grouped experts: the weight rows are [up ; gate], the result act(gate, up) as bf16 rows (GatedRows)

// bf16 products row by row up to 1024 columns and 2048 k: the weights fit an L2, and the rows are read by one XCD (us: 1280 x 1024 x 1024 20.5 -> 19.1, 517 x 1024 x 2048 19.8 -> 18.0,
// 768 x 1024 x 1536 19.9 -> 18.0; at 4096 k 517 rows 21.6 -> 22.6, f32 products of 517 x 1024 x 1024 20.9 -> 22.8).
// Where there is more than a 128 x 128 tile a CU, a last column of at most 32 behind the others while the weights are at most 48 x 1024 columns' k: 900 x 4112 x 1024 (264 tiles) 28.6 -> 27.3,
// 4000 x 4112 x 512 (1056) 47.4 -> 43.3, 2048 x 8208 x 512 (1040) 45.5 -> 41.6; of more weights 2048 x 8208 x 2048 110 -> 116, 4000 x 4112 x 2048 110 -> 115.
static TileOrder linear_tile_order(const LinearF32Params& p, uint32_t parts) {
    const uint32_t columns = (p.n + DN - 1) / DN, last = p.n % DN;
    if (columns <= 8) return parts == 1 && p.k <= 2048 ? kTileRows : kTileBlocks;
    return (p.rows + 127) / 128 * columns > 256 && last && last <= 32 && (uint64_t)columns * p.k <= 48 * 1024 ? kTileLastColumnBehind : kTileBlocks;
}

// parts: 1, or 3 for operand rows [lo | mid | hi].  partials (MB 1, not GROUPED): blockIdx.z takes its share of the k-steps and leaves its sums there, f32 [z][rows][n].
// WM x WN waves, a wave 32 MB x 64 outputs
template <int WM, int WN, int MB, int STAGES, bool GROUPED, int KIND, uint32_t parts>
__global__ void __launch_bounds__(64 * WM * WN, WM * WN == 4 ? 4 : 2) linear_dma_kernel(LinearF32Params p, const uint16_t* xb, uint32_t ldxb, GatedRows gr, float* partials, TileOrder order) {
    constexpr bool GATED = KIND == kEpilogueGated, CUT = !GROUPED && MB == 1;
    constexpr int DK = 64, DM = 32 * WM * MB, DN = 64 * WN, AP = DM * DK * 2 / 1024 / (WM * WN), BP = DN * DK * 2 / 1024 / (WM * WN); // 1 KB pieces per wave: A, B
    constexpr uint32_t STAGE = (DM + DN) * DK * 2, ROW = DK * 2, CHUNKS = DK / 8, RPP = 1024 / ROW; // row bytes, 16-byte chunks per row, rows per piece
    extern __shared__ __attribute__((aligned(1024))) uint8_t s_dma[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WN, wn = wave % WN, l32 = lane & 31, half = lane >> 5;
    uint32_t r_lo = 0, r_hi = p.rows, m_t, n_t, z = 0;
    if (GROUPED) { // tiles of the buckets back to back: the wave's lanes hold the buckets' tile counts (batch <= 64)
        const uint32_t lo = lane < p.batch ? p.row_offsets[lane] : 0u, hi = lane < p.batch ? p.row_offsets[lane + 1] : 0u;
        uint32_t upto = (hi - lo + DM - 1) / DM;
        for (uint32_t o = 1; o < 64; o <<= 1) {
            const uint32_t below = __shfl_up(upto, o, 64);
            if (lane >= o) upto += below;
        }
        const unsigned long long behind = __ballot(upto > blockIdx.y);
        if (!behind) return; // (workgroup-uniform, in front of every barrier)
        z = (uint32_t)__builtin_ctzll(behind);
        r_lo = __builtin_amdgcn_readlane(lo, z), r_hi = __builtin_amdgcn_readlane(hi, z);
        const uint32_t first = z ? __builtin_amdgcn_readlane(upto, z - 1) : 0u;
        m_t = blockIdx.y - first, n_t = blockIdx.x;
    } else {
        if (!tile_of_block(blockIdx.x, (p.rows + DM - 1) / DM, (p.n + DN - 1) / DN, order, &m_t, &n_t)) return;
    }
    const uint32_t m0 = r_lo + m_t * DM, n0 = n_t * DN;
    const uint16_t* w = p.w + (size_t)z * p.w_batch;

    // this wave's pieces of a k-step; rows outside are read from inside (never stored)
    uint32_t va[AP], vb[BP];
#pragma unroll
    for (int i = 0; i < AP; ++i) {
        const uint32_t row = (wave * AP + i) * RPP + lane / CHUNKS, chunk = (lane % CHUNKS) ^ (row >> 1 & 7);
        const uint32_t m = m0 + row < r_hi ? m0 + row : r_hi - 1;
        va[i] = (GROUPED && p.row_map ? p.row_map[m] : m) * ldxb * 2 + chunk * 16;
    }
#pragma unroll
    for (int i = 0; i < BP; ++i) {
        const uint32_t row = (wave * BP + i) * RPP + lane / CHUNKS, chunk = (lane % CHUNKS) ^ (row >> 1 & 7);
        uint32_t n = n0 + row;
        if (GATED) { // a wave's first 32 columns are up rows, its second 32 the gate rows of the same outputs: the pair meets in one lane
            const uint32_t ff = p.n / 2, f = n_t * (DN / 2) + (row >> 6) * 32 + (row & 31);
            n = (f < ff ? f : ff - 1) + (row & 32 ? ff : 0);
        } else if (n >= p.n) n = p.n - 1;
        vb[i] = n * p.k * 2 + chunk * 16;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)s_dma;
    const uint32_t w_steps = p.k / DK, all = parts * w_steps;
    const uint32_t t_lo = GROUPED ? 0u : all * blockIdx.z / gridDim.z, steps = (GROUPED ? all : all * (blockIdx.z + 1) / gridDim.z) - t_lo;
    auto fetch = [&](uint32_t step, uint32_t buf) {
        const uint32_t kt = t_lo + step, wt = parts == 1 ? kt : kt >= 2 * w_steps ? kt - 2 * w_steps : kt >= w_steps ? kt - w_steps : kt; // (the parts of a row meet the same weights)
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + buf * STAGE + wave * AP * 1024), dst_b = __builtin_amdgcn_readfirstlane(lds0 + buf * STAGE + DM * ROW + wave * BP * 1024);
        dma16<AP>(xb + kt * DK, va, dst);
        dma16<BP>(w + wt * DK, vb, dst_b);
    };

    f32x16_t acc[MB][2];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // (row_map: nothing of the compiler's is in flight from here on)
    constexpr int OPS = AP + BP; // wave-instructions of a stage
    if constexpr (STAGES > 1) {
#pragma unroll
        for (uint32_t i = 0; i + 1 < STAGES; ++i)
            if (i < steps) fetch(i, i);
    }
    uint32_t buf = 0;
    const uint32_t a_base = (wm * 32 * MB + l32) * ROW, b_base = DM * ROW + (wn * 64 + l32) * ROW, key = l32 >> 1 & 7;
    auto step = [&](uint32_t kt) {
        if constexpr (STAGES == 1) {
            if (kt) lds_barrier(); // every wave has read step kt - 1
            fetch(kt, 0);
            asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory"); // step kt is in LDS
        } else { // step kt is in LDS and every wave has read step kt - 1: step kt + STAGES - 1 may land in its place
            if (STAGES > 2 && kt + STAGES - 2 < steps) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((STAGES - 2) * OPS) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (kt + STAGES - 1 < steps) fetch(kt + STAGES - 1, buf == 0 ? STAGES - 1 : buf - 1);
        }
        const uint8_t* at = s_dma + buf * STAGE;
        if (STAGES > 1) buf = buf + 1 == STAGES ? 0 : buf + 1;
#pragma unroll
        for (uint32_t s = 0; s < DK / 16; ++s) {
            const uint32_t slot = ((2 * s + half) ^ key) * 16;
            u32x4_t af[MB], bf[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) bf[j] = *(const u32x4_t*)(at + b_base + j * 32 * ROW + slot);
#pragma unroll
            for (int i = 0; i < MB; ++i) af[i] = *(const u32x4_t*)(at + a_base + i * 32 * ROW + slot);
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, af[i]), __builtin_bit_cast(bf16x8_t, bf[j]), acc[i][j], 0, 0, 0);
        }
    };
    auto part_end = [&] { // its sums have its scale
#pragma unroll
        for (int i = 0; i < MB; ++i) acc[i][0] *= kPartDown, acc[i][1] *= kPartDown;
    };
    if constexpr (parts == 1) {
        for (uint32_t kt = 0; kt < steps; ++kt) step(kt);
    } else if constexpr (MB >= 2) { // (a loop in a loop would need the sums' registers twice)
        for (uint32_t kt = 0; kt < steps; ++kt) {
            if (t_lo + kt == w_steps || t_lo + kt == 2 * w_steps) part_end();
            step(kt);
        }
    } else {
        uint32_t kt = 0;
#pragma unroll 1
        for (uint32_t end = w_steps;; end += w_steps) {
            const uint32_t upto = end <= t_lo ? 0u : end - t_lo < steps ? end - t_lo : steps;
            for (; kt < upto; ++kt) step(kt);
            if (kt == steps) break;
            part_end();
        }
    }

    if constexpr (parts == 3) {
        if (CUT && partials) { // a share that ends inside the small parts
            const uint32_t last = t_lo + steps - 1;
            const float down = last >= 2 * w_steps ? 1.0f : last >= w_steps ? kPartDown : kPartDown * kPartDown;
#pragma unroll
            for (int i = 0; i < MB; ++i) acc[i][0] *= down, acc[i][1] *= down;
        } else {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t n = GATED ? n_t * (DN / 2) + wn * 32 + l32 : n0 + (wn * 2 + j) * 32 + l32, ends = GATED ? p.n / 2 : p.n;
                if (n >= ends) continue;
#pragma unroll
                for (int i = 0; i < MB; ++i)
                    split_repair(acc[i][j], xb, p.k, GROUPED ? p.row_map : nullptr, m0 + (wm * MB + i) * 32 + 4 * half, r_hi, w + (size_t)(GATED && j ? ends + n : n) * p.k);
            }
        }
    }
    if constexpr (GATED) {
        const uint32_t ff = p.n / 2, f = n_t * (DN / 2) + wn * 32 + l32;
        if (f >= ff) return;
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t row = m0 + (wm * MB + i) * 32 + 4 * half + (r & 3) + 8 * (r >> 2);
                if (row >= r_hi) continue;
                const float wt = gr.row_weight ? gr.row_weight[row] : 1.0f;
                const float h = expert_act(wt * acc[i][1][r], wt * acc[i][0][r], gr.act);
                if (parts == 1) gr.out[(size_t)row * ff + f] = f32_to_bf16(h);
                else {
                    uint16_t* o = gr.out + (size_t)row * 3 * ff + f;
                    split_bf16(h, o[2 * ff], o[ff], o[0]);
                }
            }
        return;
    }
    if (CUT && partials) {
        float* out = partials + (size_t)blockIdx.z * p.rows * p.n;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t n = n0 + (wn * 2 + j) * 32 + l32;
            if (n >= p.n) continue;
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t row = m0 + (wm * MB + i) * 32 + 4 * half + (r & 3) + 8 * (r >> 2);
                    if (row < r_hi) out[(size_t)row * p.n + n] = acc[i][j][r];
                }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uint32_t n = n0 + (wn * 2 + j) * 32 + l32;
        if (n >= p.n) continue;
        const float bias = p.bias ? bf16_to_f32(p.bias[n]) : 0.0f;
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            const uint32_t row0 = m0 + (wm * MB + i) * 32 + 4 * half;
            float res[16]; // (the residual may be y itself: a block's rows are read before any of them is stored)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t row = row0 + (r & 3) + 8 * (r >> 2);
                res[r] = p.residual && row < r_hi ? p.residual[(size_t)row * p.ldr + n] : 0.0f;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t row = row0 + (r & 3) + 8 * (r >> 2);
                if (row >= r_hi) continue;
                const float v = linear_value<KIND>(acc[i][j][r], bias, p, row, z, n);
                p.y[(size_t)row * p.ldy + n] = p.residual ? v + res[r] : v;
            }
        }
    }
}

// f32 rows -> bf16 rows, round to nearest even: what the product's operand is
__global__ void __launch_bounds__(256) linear_bf16_rows_kernel(const float* x, uint32_t ldx, uint16_t* out, uint32_t k, size_t chunks) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; // chunk of 8
    if (i >= chunks) return;
    const uint32_t per_row = k / 8;
    const size_t r = i / per_row;
    const uint32_t c = (uint32_t)(i - r * per_row) * 8;
    const f32x4_v a = *(const f32x4_v*)(x + r * ldx + c), b = *(const f32x4_v*)(x + r * ldx + c + 4);
    u32x4_v o;
    o.x = pack_bf16(a.x, a.y), o.y = pack_bf16(a.z, a.w), o.z = pack_bf16(b.x, b.y), o.w = pack_bf16(b.z, b.w);
    *(u32x4_v*)(out + i * 8) = o;
}

// ... and the rows [lo | mid | hi] of 3 k
__global__ void __launch_bounds__(256) linear_split_rows_kernel(const float* x, uint32_t ldx, uint16_t* out, uint32_t k, size_t chunks) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; // chunk of 4
    if (i >= chunks) return;
    const uint32_t per_row = k / 4;
    const size_t r = i / per_row;
    const uint32_t c = (uint32_t)(i - r * per_row) * 4;
    const f32x4_v a = *(const f32x4_v*)(x + r * ldx + c);
    uint16_t h[4], m[4], l[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) split_bf16(a[j], h[j], m[j], l[j]);
    uint16_t* o = out + r * 3 * k + c;
    auto put = [](uint16_t* at, const uint16_t (&v)[4]) { *(u32x2_v*)at = u32x2_v{(uint32_t)v[0] | ((uint32_t)v[1] << 16), (uint32_t)v[2] | ((uint32_t)v[3] << 16)}; };
    put(o, l), put(o + k, m), put(o + 2 * k, h);
}

// the shares of a product cut along k, added in their order, and the product's end
template <uint32_t PARTS> __global__ void __launch_bounds__(256) linear_finish_kernel(LinearF32Params p, const uint16_t* xb, const float* partials, uint32_t splits) {
    const size_t total = (size_t)p.rows * p.n, i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    float sum = partials[i];
    for (uint32_t z = 1; z < splits; ++z) sum += partials[z * total + i];
    const uint32_t row = (uint32_t)(i / p.n), n = (uint32_t)(i - (size_t)row * p.n);
    if (PARTS == 3 && sum != sum) sum = split_dot(xb + (size_t)row * 3 * p.k, p.w + (size_t)n * p.k, p.k);
    p.y[(size_t)row * p.ldy + n] = linear_epilogue(sum, p.bias ? bf16_to_f32(p.bias[n]) : 0.0f, p, row, 0, n);
}

template <int WM, int WN, int MB, int STAGES, bool GROUPED, int KIND, uint32_t PARTS>
uzu_status launch_dma_tile(hipStream_t s, const LinearF32Params& p, const uint16_t* xb, const GatedRows& gr, float* partials, uint32_t splits) {
    constexpr uint32_t DM = 32 * WM * MB, TN = 64 * WN;
    const uint32_t m_tiles = (p.rows + DM - 1) / DM, n_tiles = (p.n + TN - 1) / TN;
    const dim3 grid = GROUPED ? dim3(n_tiles, m_tiles + p.batch) : dim3(tile_order_grid(m_tiles, n_tiles), 1, splits);
    UZU_REQUIRE(grid.y <= 65535, "linear_dma: grid too large");
    const size_t lds = (size_t)STAGES * (DM + TN) * 64 * 2;
    static LdsLimit lim;
    UZU_REQUIRE(raise_lds_limit(lim, (const void*)linear_dma_kernel<WM, WN, MB, STAGES, GROUPED, KIND, PARTS>, lds), "linear_dma: %zu bytes of LDS are not available", lds);
    return launch_check([&] { hipLaunchKernelGGL((linear_dma_kernel<WM, WN, MB, STAGES, GROUPED, KIND, PARTS>), grid, dim3(64 * WM * WN), lds, s, p, xb, PARTS * p.k, gr, partials, linear_tile_order(p, PARTS)); }, "linear_dma");
}
template <bool GROUPED, int KIND, uint32_t PARTS> uzu_status launch_dma(hipStream_t s, const LinearF32Params& p, const uint16_t* xb, const GatedRows& gr = GatedRows()) {
    const size_t tiles = (size_t)((p.rows + 127) / 128) * ((p.n + DN - 1) / DN);
    if (tiles >= 512) return launch_dma_tile<2, 2, 2, 1, GROUPED, KIND, PARTS>(s, p, xb, gr, nullptr, 1);
    if (tiles > 256) return launch_dma_tile<2, 2, 2, 2, GROUPED, KIND, PARTS>(s, p, xb, gr, nullptr, 1);
    return launch_dma_tile<2, 2, 1, 2, GROUPED, KIND, PARTS>(s, p, xb, gr, nullptr, 1);
}
// Few tiles, many k-steps: the steps are cut over workgroups (two a CU wanted, eight steps each at least) and the shares added by a launch of their own.
// 300 x 1024 x 2048: f32 products 56 us in one piece and 21.8 us cut (VALU tile: 217 us), bf16 products 26.5 us in the register-staged form and 16.0 us.
uint32_t dma_splits(const LinearF32Params& p, uint32_t parts) {
    const uint32_t tiles = ((p.rows + 63) / 64) * ((p.n + DN - 1) / DN), steps = parts * p.k / 64;
    uint32_t splits = 1;
    while (splits < 8 && tiles * splits * 2 <= 512 && steps >= 16 * splits) splits *= 2;
    return splits;
}
// Up to a 128 x 128 tile a CU: eight waves on it (32 x 64 outputs each) over four buffers of one k-step, and K cut until there is about a workgroup a CU, eight steps each at least;
// 0: not this form.  Against the 64-row tiles, us: 2048 x 2048 x 4096 70 -> 53, 1000 x 2048 x 4096 46 -> 36 (two shares), 517 x 2048 x 4096 38.5 -> 27.9 (three), 300 x 7712 x 2048
// 37 -> 29; f32 products 517 x 2048 x 4096 74 -> 50, 300 x 2048 x 4096 44 -> 36.  Those stay ahead where half of these tiles' rows would be empty and there are many of them
// (64 x 7712 x 2048 18.8 against 20.2), where the steps allow no more than half of the chip (1000 x 1024 x 1024 18 against 20) and where they cut an f32 product that this form cannot
// (400 x 4112 x 1024 29 against 37).
uint32_t eight_wave_splits(const LinearF32Params& p, uint32_t parts) {
    const uint32_t tiles = ((p.rows + 127) / 128) * ((p.n + 127) / 128), steps = parts * p.k / 64;
    if (tiles > 256 || (p.rows <= 64 && tiles > 48)) return 0;
    // (an XCD of 32 CUs has an eighth of a share's tiles, rounded up: seven shares of 36 tiles are 35 workgroups on some, two rounds: 768 x 768 x 4096 29.9 us, in six shares 24.1)
    uint32_t splits = std::min(8u, 32 / ((tiles + 7) / 8));
    while (splits > 1 && steps < 8 * splits) --splits;
    if (tiles >= 64 && tiles * splits <= 128) return 0;
    return parts == 3 && splits == 1 && dma_splits(p, parts) > 1 ? 0 : splits;
}
// the operand rows and, behind them, the shares of a cut product
size_t dma_workspace(const LinearF32Params& p, uint32_t parts) {
    const uint32_t splits = std::max(dma_splits(p, parts), eight_wave_splits(p, parts));
    return ((size_t)p.rows * p.k * 2 * parts + 255) / 256 * 256 + (splits > 1 ? (size_t)splits * p.rows * p.n * 4 : 0);
}
template <uint32_t PARTS> uzu_status launch_dma_plain(hipStream_t s, const LinearF32Params& p, uint16_t* ws) {
    float* partials = (float*)((char*)ws + ((size_t)p.rows * p.k * 2 * PARTS + 255) / 256 * 256);
    const uint32_t eight = eight_wave_splits(p, PARTS);
    if (const uint32_t splits = eight ? eight : dma_splits(p, PARTS); splits > 1) {
        if (eight) UZU_PROPAGATE((launch_dma_tile<4, 2, 1, 4, false, kEpilogueLean, PARTS>(s, p, ws, GatedRows(), partials, splits)));
        else UZU_PROPAGATE((launch_dma_tile<2, 2, 1, 2, false, kEpilogueLean, PARTS>(s, p, ws, GatedRows(), partials, splits)));
        const size_t total = (size_t)p.rows * p.n;
        return launch_check([&] { hipLaunchKernelGGL(linear_finish_kernel<PARTS>, dim3((uint32_t)((total + 255) / 256)), dim3(256), 0, s, p, ws, partials, splits); }, "linear_finish");
    }
    if (eight) {
        switch (epilogue_kind(p)) {
        case kEpilogueLean: return launch_dma_tile<4, 2, 1, 4, false, kEpilogueLean, PARTS>(s, p, ws, GatedRows(), nullptr, 1);
        case kEpilogueXielu: return launch_dma_tile<4, 2, 1, 4, false, kEpilogueXielu, PARTS>(s, p, ws, GatedRows(), nullptr, 1);
        default: return launch_dma_tile<4, 2, 1, 4, false, kEpilogueFull, PARTS>(s, p, ws, GatedRows(), nullptr, 1);
        }
    }
    switch (epilogue_kind(p)) {
    case kEpilogueLean: return launch_dma<false, kEpilogueLean, PARTS>(s, p, ws);
    case kEpilogueXielu: return launch_dma<false, kEpilogueXielu, PARTS>(s, p, ws);
    default: return launch_dma<false, kEpilogueFull, PARTS>(s, p, ws);
    }
}

// Shapes with whole k-steps.  The form is three short launches (operand rows, tiles, shares), 12 us at the least.  bf16 products (parts 1): the register-staged form takes
// 9.5 us at k = 512, 15 us at k = 1024, 26 us at k = 2048 whatever the rows, until there are tiles for the whole chip (2 GFLOP).  Up to 64 rows it takes 64 columns a workgroup where this
// form's tiles have 128, and is ahead over wide outputs of short contractions unless this form's last round of tiles, four a CU, is full: 49152 x 1024 (384 tiles) 24 us against 30 at 64 rows,
// 65536 x 1024 (512) 34 against 38, 151936 x 1024 (1187) 90 against 101, but 131072 x 1024 (1024) 83 against 70 and 32768 x 2048 45 against 40.  f32 products (parts 3): the VALU tile takes
// 0.1 us per k-step of one (55 us at k = 512, 217 us at k = 2048) against 14 to 22 us.
bool dma_shape(uint32_t rows, uint32_t n, uint32_t k, uint32_t parts) {
    const double gflops = 2e-9 * rows * n * k;
    if (n < 64 || k % 64 || (uint64_t)rows * k * parts * 2 >= 1ull << 32 || (uint64_t)n * k * 2 >= 1ull << 32) return false; // (32-bit byte offsets)
    if (parts == 1 && rows <= 64 && n >= 32768 && k < 2048) {
        const uint32_t tiles = (n + DN - 1) / DN, last = tiles % 1024;
        if (last && last < 920) return false;
    }
    return rows > 16 && (parts == 1 ? (rows >= 128 && gflops >= 2.0) || k >= 1024 : k >= 256 || gflops >= 0.05);
}

template <int MB, int NB> uzu_status launch(hipStream_t s, const LinearF32Params& p, const char* what) {
    const dim3 grid((p.n + 64 * NB - 1) / (64 * NB), (p.rows + 64 * MB - 1) / (64 * MB), p.batch);
    UZU_REQUIRE(grid.y <= 65535 && grid.z <= 65535, "linear_mfma: grid too large");
    switch (epilogue_kind(p)) {
    case kEpilogueLean: return launch_check([&] { hipLaunchKernelGGL((linear_mfma_kernel<MB, NB, false, kEpilogueLean>), grid, dim3(256), 0, s, p); }, what);
    case kEpilogueXielu: return launch_check([&] { hipLaunchKernelGGL((linear_mfma_kernel<MB, NB, false, kEpilogueXielu>), grid, dim3(256), 0, s, p); }, what);
    default: return launch_check([&] { hipLaunchKernelGGL((linear_mfma_kernel<MB, NB, false, kEpilogueFull>), grid, dim3(256), 0, s, p); }, what);
    }
}

} // namespace

bool linear_mfma_supported(const LinearF32Params& p) {
    if (!p.bf16_products || (p.rows <= 16 && !p.row_offsets) || p.k % 8 || p.ldx % 4 || p.x_batch % 4 || p.w_batch % 8) return false;
    if ((uintptr_t)p.x % 16 || (uintptr_t)p.w % 16) return false;
    if (p.row_offsets && ((uint64_t)p.rows * p.ldx >= 1ull << 32 || (uint64_t)p.n * p.k >= 1ull << 32)) return false; // (grouped: element offsets inside a product are 32-bit)
    return true;
}

uzu_status linear_bf16_rows(hipStream_t s, const float* x, uint32_t ldx, uint16_t* out, uint32_t rows, uint32_t k) {
    const size_t chunks = (size_t)rows * (k / 8);
    UZU_REQUIRE(k % 8 == 0 && ldx % 4 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)out & 15) == 0, "linear_bf16_rows: alignment");
    return launch_check([&] { hipLaunchKernelGGL(linear_bf16_rows_kernel, dim3((uint32_t)((chunks + 255) / 256)), dim3(256), 0, s, x, ldx, out, k, chunks); }, "linear_bf16_rows");
}
uzu_status linear_split_rows(hipStream_t s, const float* x, uint32_t ldx, uint16_t* out, uint32_t rows, uint32_t k) {
    const size_t chunks = (size_t)rows * (k / 4);
    UZU_REQUIRE(k % 4 == 0 && ldx % 4 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)out & 15) == 0, "linear_split_rows: alignment");
    return launch_check([&] { hipLaunchKernelGGL(linear_split_rows_kernel, dim3((uint32_t)((chunks + 255) / 256)), dim3(256), 0, s, x, ldx, out, k, chunks); }, "linear_split_rows");
}
bool linear_dma_grouped_supported(const LinearF32Params& p) {
    return p.row_offsets && p.batch <= 64 && !p.residual && epilogue_kind(p) == kEpilogueLean && p.w_batch % 8 == 0 && ((uintptr_t)p.w & 15) == 0 &&
           dma_shape(p.rows, p.n, p.k, p.bf16_products ? 1 : 3);
}
uzu_status linear_dma_grouped(hipStream_t s, const LinearF32Params& p, const uint16_t* xb, const GatedRows* gated) {
    UZU_REQUIRE(linear_dma_grouped_supported(p) && ((uintptr_t)xb & 15) == 0 && (!gated || (gated->out && p.n % 2 == 0 && !p.bias)), "linear_dma_grouped: shape / alignment not covered");
    if (p.bf16_products) return gated ? launch_dma<true, kEpilogueGated, 1>(s, p, xb, *gated) : launch_dma<true, kEpilogueLean, 1>(s, p, xb);
    return gated ? launch_dma<true, kEpilogueGated, 3>(s, p, xb, *gated) : launch_dma<true, kEpilogueLean, 3>(s, p, xb);
}
// f32 products of enough rows: false = not covered (or no workspace: the stream is captured), nothing launched
bool linear_split(hipStream_t s, const LinearF32Params& p, uzu_status* st) {
    if (p.bf16_products || p.row_offsets || p.row_map || p.batch != 1 || p.ldx % 4 || (((uintptr_t)p.x | (uintptr_t)p.w) & 15) || !dma_shape(p.rows, p.n, p.k, 3)) return false;
    uint16_t* xb = (uint16_t*)stream_workspace(s, dma_workspace(p, 3));
    if (!xb) return false;
    *st = linear_split_rows(s, p.x, p.ldx, xb, p.rows, p.k);
    if (*st == UZU_OK) *st = launch_dma_plain<3>(s, p, xb);
    return true;
}

uzu_status linear_mfma(hipStream_t s, const LinearF32Params& p) {
    UZU_REQUIRE(linear_mfma_supported(p), "linear_mfma: shape / alignment not covered");
    UZU_REQUIRE(p.row_offsets || !p.row_map, "linear_mfma: gathered rows only in the grouped form");
    if (!p.row_offsets && p.batch == 1 && dma_shape(p.rows, p.n, p.k, 1)) {
        if (uint16_t* xb = (uint16_t*)stream_workspace(s, dma_workspace(p, 1))) { // (none while the stream is captured)
            UZU_PROPAGATE(linear_bf16_rows(s, p.x, p.ldx, xb, p.rows, p.k));
            return launch_dma_plain<1>(s, p, xb);
        }
    }
    // tile choice: the widest tile that still fills the chip; narrow outputs (the per-head products) take the narrow tiles
    if (p.row_offsets) { // grouped: every product may need the whole row range, the workgroups beyond a bucket leave at once
        const dim3 grid((p.n + 127) / 128, (p.rows + 127) / 128 + 1, p.batch);
        UZU_REQUIRE(grid.y <= 65535 && grid.z <= 65535 && !p.residual && epilogue_kind(p) == kEpilogueLean, "linear_mfma: a grouped launch of that size, with a residual or more than a bias and an activation");
        return launch_check([&] { hipLaunchKernelGGL((linear_mfma_kernel<2, 2, true, kEpilogueLean>), grid, dim3(256), 0, s, p); }, "linear_mfma_grouped");
    }
    const bool small_m = p.rows <= 64, small_n = p.n <= 64;
    auto tiles = [&](uint32_t bm, uint32_t bn) { return (size_t)((p.rows + bm - 1) / bm) * ((p.n + bn - 1) / bn) * p.batch; };
    if (!small_m && !small_n && tiles(128, 128) >= 256) return launch<2, 2>(s, p, "linear_mfma<2,2>");
    if (!small_m && (small_n || tiles(128, 64) >= 256)) return launch<2, 1>(s, p, "linear_mfma<2,1>");
    return launch<1, 1>(s, p, "linear_mfma<1,1>");
}

} // namespace k
} // namespace uzu
