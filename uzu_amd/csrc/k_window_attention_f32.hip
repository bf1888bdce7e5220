// k_window_attention_f32.hip -- prompt attention over caches of f32 rows on the f32 matrix cores, for the f32-stream designs (kernels_stream32.h: WindowAttentionParams).
//
// What bounds it: at a few hundred rows the way from the first load to the last sum; the simple form (a wave per row and head, k_window_attention.hip) reads every key and value once per row
// and spends an addition of a lane on each product.  Here a workgroup has 16 rows of a head, and its eight waves share the blocks of 16 keys by the block's number, each with its own running
// maximum and sums, which meet in LDS at the end, in wave order: no barrier before.  v_mfma_f32_16x16x4_f32: products and sums in f32, as the simple form's.
//   scores   S^T = K Q^T: a lane holds four keys' scores of one query (key 4 (lane / 16) + r, query lane % 16), and its softmax statistics
//   results  O^T = V^T P^T: step s takes the keys 4 (lane / 16) + s, whose weights are the lane's own registers; the queries stay where they are
// Keys and values go from memory into the operands' registers, a wave's next ones while it works.  A block's number counts from position 0, and a key that a row does not see has weight 0: a row's
// sums do not depend on what else is in its tile or its pass.  (Zero times a value that is not finite is no zero: where that shows, a row's sums are made again from its keys alone.)
// 300 rows of 8 heads of 128: 44.7 us by the simple form, 15.3 here.  (29.5 with a branch around every load for caches of four bytes' alignment, which the loads take as they are, and with the
// values, too, a step ahead, which spilled.)
#include "device_utils.h"
#include "kernels_stream32.h"

namespace uzu {
namespace k {

namespace {
constexpr uint32_t kRows = 16, kKeys = 16, kWaves = 8;

// Columns c .. c + 3 of a row's sums, those that are NaN, from the keys that the row (position t) sees, one after the other
template <bool EXTRA>
__device__ __forceinline__ void visible_sums(const WindowAttentionParams& p, size_t row, uint32_t t, uint32_t a, const float* K, const float* V, size_t kpitch, size_t vpitch, uint32_t dim, uint32_t c,
                                          float top, f32x4_v& v) {
    const float *q = p.q + row * p.ldq + (size_t)a * dim, hscale = p.head_scale ? p.scale * p.head_scale[a] : p.scale;
    uint32_t j = p.window && t + 1 > p.window ? t + 1 - p.window : 0u;
    f32x4_v sums = {0.f, 0.f, 0.f, 0.f};
    for (j = p.chunk ? max(j, t / p.chunk * p.chunk) : j; j <= t; ++j) {
        float s = 0.0f;
        for (uint32_t i = 0; i < dim; ++i) s = fmaf(K[j * kpitch + i], q[i], s);
        s *= hscale;
        if (EXTRA && p.soft_cap != 0.0f) s = p.soft_cap * tanhf(s / p.soft_cap);
        if (EXTRA && p.dist_bias) s += p.dist_bias[(size_t)min(t - j, p.dist_rows - 1) * p.heads + a];
        const float w = expf(s - top);
        for (uint32_t e = 0; e < 4; ++e) sums[e] = fmaf(w, V[j * vpitch + c + e], sums[e]);
    }
    for (uint32_t e = 0; e < 4; ++e) v[e] = v[e] != v[e] ? sums[e] : v[e];
}

// grid (row tiles at most, heads), 512 threads.  DG: key width / 16; VH: value width / 64
// EXTRA: a cap on the scores or a bias by distance (an instance of its own: the plain one has no branch between the products)
template <int DG, int VH, bool EXTRA>
__global__ void __launch_bounds__(64 * kWaves) window_attention_f32_kernel(WindowAttentionParams p) {
    constexpr int DIM = 16 * DG, VD = 64 * VH, OP = VD + 4;
    __shared__ __attribute__((aligned(16))) float s_o[kWaves][kRows][OP];
    __shared__ float s_m[kWaves][kRows], s_l[kWaves][kRows];
    const uint32_t tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, kq = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6), a = blockIdx.y, g = a / (p.heads / p.kv_heads);
    uint32_t tile = blockIdx.x, z = 0;
    SeqSpan sp;
    for (;; ++z) { // the tile's sequence
        if (z == p.nseq) return;
        sp = p.spans[z];
        const uint32_t n = (sp.count + kRows - 1) / kRows;
        if (tile < n) break;
        tile -= n;
    }
    const uint32_t row0 = tile * kRows, rows = min(sp.count - row0, kRows), r = sp.row0 + row0 + min(l16, rows - 1), t = sp.start + row0 + min(l16, rows - 1); // (rows past the last: the last again)
    auto first_key = [&](uint32_t at) {
        uint32_t lo = p.window && at + 1 > p.window ? at + 1 - p.window : 0u;
        return p.chunk ? max(lo, at / p.chunk * p.chunk) : lo;
    };
    const uint32_t lo = first_key(t), last = sp.start + row0 + rows - 1, block0 = first_key(sp.start + row0) / kKeys, block1 = last / kKeys; // (the first row sees furthest back)
    const float* K = (const float*)p.key_caches[z] + (size_t)g * DIM;
    const float* V = (const float*)p.value_caches[z] + (size_t)g * VD;
    const size_t kpitch = (size_t)p.kv_heads * DIM, vpitch = (size_t)p.kv_heads * VD;
    typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4))); // (global loads of four words want aligned words)
    auto load4 = [](const float* at) { return (f32x4_v)*(const f32x4_u*)at; };
    f32x4_v keys[DG], next[DG], values[4][VH];
    auto load_keys = [&](uint32_t block, f32x4_v (&to)[DG]) {
        const float* row = K + (size_t)min(block * kKeys + l16, last) * kpitch + 4 * kq;
#pragma unroll
        for (int i = 0; i < DG; ++i) to[i] = load4(row + 16 * i);
    };
    auto load_values = [&](uint32_t block, f32x4_v (&to)[4][VH]) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float* row = V + (size_t)min(block * kKeys + 4 * kq + s, last) * vpitch + 4 * l16;
#pragma unroll
            for (int h = 0; h < VH; ++h) to[s][h] = load4(row + 64 * h);
        }
    };
    uint32_t block = block0 + ((wave - block0) & (kWaves - 1)); // this wave's first: its number in the last three bits
    if (block <= block1) load_keys(block, keys);
    f32x4_v qf[DG];
    const float* q = p.q + (size_t)r * p.ldq + (size_t)a * DIM + 4 * kq;
#pragma unroll
    for (int i = 0; i < DG; ++i) qf[i] = *(const f32x4_v*)(q + 16 * i);
    const float hscale = p.head_scale ? p.scale * p.head_scale[a] : p.scale;

    f32x4_v o[VH][4];
#pragma unroll
    for (int h = 0; h < VH; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[h][e] = f32x4_v{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.0f; // l: this lane's keys
    for (; block <= block1; block += kWaves) {
        load_values(block, values);
        load_keys(min(block + kWaves, block1), next);
        __builtin_amdgcn_sched_barrier(0);
        f32x4_v part[4] = {}; // (four chains)
#pragma unroll
        for (int i = 0; i < DG; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) part[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(keys[i][e], qf[i][e], part[e], 0, 0, 0);
        const f32x4_v dot = (part[0] + part[1]) + (part[2] + part[3]);
        float w[4], m_new = m;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t j = block * kKeys + 4 * kq + i;
            float s = dot[i] * hscale;
            if constexpr (EXTRA)
                if (p.soft_cap != 0.0f) s = p.soft_cap * tanhf(s / p.soft_cap);
            if (j < lo || j > t) s = -INFINITY;
            else if (EXTRA && p.dist_bias) s += p.dist_bias[(size_t)min(t - j, p.dist_rows - 1) * p.heads + a];
            w[i] = s;
            m_new = fmaxf(m_new, s);
        }
        m_new = fmaxf(m_new, __shfl_xor(m_new, 16, 64)), m_new = fmaxf(m_new, __shfl_xor(m_new, 32, 64));
        const float corr = m_new == m ? 1.0f : expf(m - m_new); // (first keys: 0)
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = w[i] == -INFINITY ? 0.0f : expf(w[i] - m_new);
        l = l * corr + ((w[0] + w[1]) + (w[2] + w[3])), m = m_new;
#pragma unroll
        for (int h = 0; h < VH; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                o[h][e] *= corr;
#pragma unroll
                for (int s = 0; s < 4; ++s) o[h][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(values[s][h][e], w[s], o[h][e], 0, 0, 0);
            }
#pragma unroll
        for (int i = 0; i < DG; ++i) keys[i] = next[i];
    }
    l += __shfl_xor(l, 16, 64), l += __shfl_xor(l, 32, 64);
    if (kq == 0) s_m[wave][l16] = m, s_l[wave][l16] = l;
#pragma unroll
    for (int h = 0; h < VH; ++h) // tile (h, e): column 64 h + 4 (4 kq + r) + e
#pragma unroll
        for (int i = 0; i < 4; ++i) *(f32x4_v*)&s_o[wave][l16][64 * h + 16 * kq + 4 * i] = f32x4_v{o[h][0][i], o[h][1][i], o[h][2][i], o[h][3][i]};
    __syncthreads();
    // the waves' sums, in wave order: a thread has four columns of a row
    const uint32_t row = tid & 15, c = (tid >> 4) * 4;
    if (row >= rows || c >= VD) return;
    float all = p.sinks ? p.sinks[a] : -INFINITY, sum = 0.0f;
#pragma unroll
    for (uint32_t w = 0; w < kWaves; ++w) all = fmaxf(all, s_m[w][row]);
    f32x4_v v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (uint32_t w = 0; w < kWaves; ++w) {
        const float f = s_m[w][row] == -INFINITY ? 0.0f : expf(s_m[w][row] - all);
        sum += s_l[w][row] * f, v += *(const f32x4_v*)&s_o[w][row][c] * f;
    }
    if (p.sinks) sum += expf(p.sinks[a] - all);
    const size_t out_row = sp.row0 + row0 + row;
    const f32x4_v lost = v - v; // (NaN or zero)
    if (__builtin_expect(((lost[0] + lost[1]) + (lost[2] + lost[3])) != 0.0f && sum == sum, 0)) visible_sums<EXTRA>(p, out_row, sp.start + row0 + row, a, K, V, kpitch, vpitch, DIM, c, all, v);
    const float og = p.gate ? p.out_scale / (1.0f + expf(-p.gate[out_row * p.ldgate + a])) : p.out_scale;
    float* out = p.out + out_row * p.ldo + (size_t)a * VD + c;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = v[e] / sum * og;
}
} // namespace

// Short windows and few rows are left to the simple form: a wave has few keys there, and a tile of sixteen rows has the windows of all of them.  Us, simple and here: 8 heads of 128, window 64, 16 / 64 /
// 100 rows 6.8 / 9.7, 7.6 / 9.7, 9.4 / 9.9; window 128, 48 rows 11.3 / 11.7; 16 heads, window 64, 64 / 100 rows 9.5 / 9.9, 12.6 / 10.0; 32 heads of 64, window 64, 32 rows 6.8 / 6.7; window 192 is here always.
bool window_attention_f32_supported(const WindowAttentionParams& p) {
    if (p.window && p.window <= 128 && (uint64_t)p.rows * p.heads * p.window <= 65536) return false;
    return !p.cache_bf16 && (p.dim == 64 || p.dim == 128) && (p.vdim == 64 || p.vdim == 128) && p.nseq && p.rows >= kRows * p.nseq && p.ldq % 4 == 0 && ((uintptr_t)p.q & 15) == 0 && p.heads <= 65535;
}

uzu_status window_attention_f32(hipStream_t s, const WindowAttentionParams& p) {
    const dim3 grid(p.rows / kRows + p.nseq, p.heads); // (a sequence's last tile may be a part of one)
    const bool extra = p.soft_cap != 0.0f || p.dist_bias;
    return launch_check([&] {
#define UZU_WF(DG, VH)                                                                                                            \
    if (extra) hipLaunchKernelGGL((window_attention_f32_kernel<DG, VH, true>), grid, dim3(64 * kWaves), 0, s, p);                 \
    else hipLaunchKernelGGL((window_attention_f32_kernel<DG, VH, false>), grid, dim3(64 * kWaves), 0, s, p)
        if (p.dim == 64 && p.vdim == 64) {
            UZU_WF(4, 1);
        } else if (p.dim == 64) {
            UZU_WF(4, 2);
        } else if (p.vdim == 64) {
            UZU_WF(8, 1);
        } else {
            UZU_WF(8, 2);
        }
#undef UZU_WF
    }, "window_attention_f32");
}

} // namespace k
} // namespace uzu
