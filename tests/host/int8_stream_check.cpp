// The stream of large int8 matrices (k_decode_large.hip) on the GPU, bit for bit what the decode GEMV's own kernels (k_decode.hip) make of the same rows, which they get in parts too small for the
// stream: one and two matrices, up / gate pairs, with and without the Normalization in front, biases and the read-out's arg-max; rows that do not divide by the waves, the shortest and the longest
// row, and three items of a wave on their way (from 128 MB on).
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../uzu_amd/csrc/kernels.h"
#include "../../uzu_amd/csrc/kernels_decode.h"
#include "../../uzu_amd/csrc/uzu_math.h"

using namespace uzu;

constexpr int kCus = 256;

static void hip(hipError_t e) {
    if (e != hipSuccess) printf("%s\n", hipGetErrorString(e)), exit(2);
}
template <class T> static T* device(size_t count) {
    T* p = nullptr;
    hip(hipMalloc((void**)&p, count * sizeof(T)));
    return p;
}
template <class T> static T* upload(const std::vector<T>& v) {
    T* p = device<T>(v.size());
    hip(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return p;
}
template <class T> static std::vector<T> download(const T* p, size_t count) {
    std::vector<T> v(count);
    hip(hipMemcpy(v.data(), p, count * sizeof(T), hipMemcpyDeviceToHost));
    return v;
}
static uint32_t run(const k::DecGemvParams& p) {
    uint32_t grid = 0;
    if (k::gemv_dec(nullptr, p, kCus, &grid) != UZU_OK) printf("%s\n", uzu_hip_last_error()), exit(2);
    hip(hipDeviceSynchronize());
    return grid;
}

int main() {
    struct Case {
        uint32_t k, n0, n1, group;
        bool norm, act, bias, amax;
    };
    std::mt19937 rng(3);
    std::normal_distribution<float> normal;
    int bad = 0;
    for (const Case& c : {Case{2048, 4099, 0, 128, false, false, true, false}, {2048, 6410, 0, 32, true, true, true, false}, {2048, 3003, 1501, 64, true, false, true, false}, {4096, 3001, 0, 128, true, false, false, true},
                          {6144, 2222, 0, 2048, true, true, false, false}, {8192, 2060, 0, 64, true, true, false, false}, {8192, 16401, 0, 128, true, false, false, true}, {10240, 835, 0, 32, false, false, false, true},
                          {14336, 300, 333, 128, false, false, false, false}, {32768, 263, 0, 128, false, false, true, false}}) {
        const uint32_t k = c.k, rows = c.n0 + c.n1, groups = k / c.group;
        std::vector<uint8_t> w((size_t)rows * k);
        for (size_t i = 0; i < w.size(); i += 4) {
            const uint32_t r = rng();
            w[i] = r, w[i + 1] = r >> 8, w[i + 2] = r >> 16, w[i + 3] = r >> 24;
        }
        auto random = [&](size_t count, float mean, float size) {
            std::vector<uint16_t> v(count);
            for (uint16_t& x : v) x = f32_to_bf16(mean + size * normal(rng));
            return v;
        };
        std::vector<float> norm(k);
        for (float& x : norm) x = 1.0f + 0.1f * normal(rng);
        uint8_t* d_w = upload(w);
        uint16_t *d_s = upload(random((size_t)rows * groups, 0.01f, 0.002f)), *d_o = upload(random((size_t)rows * groups, -1.28f, 0.1f)), *d_b = upload(random(rows, 0.0f, 1.0f));
        k::DecGemvParams p{};
        p.k = k, p.bits = 8, p.group_size = c.group, p.b_kind = UZU_MATMUL_B_SCALE_BIAS, p.x = upload(random(k, 0.0f, 1.0f));
        if (c.norm) p.norm_scales = upload(norm), p.norm_eps = 1e-5f, p.norm_full_layer = 1, p.residual_add = 1, p.shortcut_in = upload(random(k, 0.0f, 1.0f)), p.shortcut_out = device<uint16_t>(k), p.normed_out = device<uint16_t>(k);
        p.act_mul = c.act;
        auto bind = [&](k::DecGemvParams& q, int m, const uint8_t* weights, size_t first, uint32_t count, const uint16_t* s, const uint16_t* o, const uint16_t* b, uint16_t* out) {
            q.w[m] = weights + first * k, q.scales[m] = s + first * groups, q.biases[m] = o + first * groups, q.out_bias[m] = c.bias ? b + first : nullptr, q.n[m] = count, q.out[m] = out;
        };
        uint16_t *whole = device<uint16_t>(rows), *parts = device<uint16_t>(rows);
        k::DecGemvParams q = p;
        bind(q, 0, d_w, 0, c.n0, d_s, d_o, d_b, whole);
        if (c.n1) bind(q, 1, d_w, c.n0, c.n1, d_s, d_o, d_b, whole + c.n0);
        float* top_value = device<float>(8192);
        uint32_t* top_index = device<uint32_t>(8192);
        if (c.amax) q.part_val = top_value, q.part_idx = top_index, q.part_capacity = 8192;
        if (!k::gemv_large_wanted(q, kCus)) printf("K = %u: not for the stream\n", k), ++bad;
        const uint32_t grid = run(q);
        std::vector<uint16_t> row_out[2][2];
        if (c.norm) row_out[0][0] = download(p.shortcut_out, k), row_out[0][1] = download(p.normed_out, k);
        // the same rows in parts of less than 8 MB (pairs: their up rows, then their gate rows)
        const uint32_t results = c.act ? c.n0 / 2 : rows, most = 1000 * 2048 / k * (c.act ? 2 : 4) / 2;
        uint8_t* part_w = device<uint8_t>((size_t)2 * most * k);
        uint16_t *part_s = device<uint16_t>((size_t)2 * most * groups), *part_o = device<uint16_t>((size_t)2 * most * groups), *part_b = device<uint16_t>(2 * most);
        for (uint32_t first = 0; first < results; first += most) {
            const uint32_t count = std::min(most, results - first);
            q = p;
            if (c.act) {
                for (uint32_t h = 0; h < 2; ++h) {
                    const size_t from = first + (h ? results : 0u), to = h * count;
                    hip(hipMemcpy(part_w + to * k, d_w + from * k, (size_t)count * k, hipMemcpyDeviceToDevice));
                    hip(hipMemcpy(part_s + to * groups, d_s + from * groups, (size_t)count * groups * 2, hipMemcpyDeviceToDevice));
                    hip(hipMemcpy(part_o + to * groups, d_o + from * groups, (size_t)count * groups * 2, hipMemcpyDeviceToDevice));
                    hip(hipMemcpy(part_b + to, d_b + from, (size_t)count * 2, hipMemcpyDeviceToDevice));
                }
                bind(q, 0, part_w, 0, 2 * count, part_s, part_o, part_b, parts + first);
            } else {
                bind(q, 0, d_w, first, count, d_s, d_o, d_b, parts + first);
            }
            if (k::gemv_large_wanted(q, kCus)) printf("K = %u: a part for the stream\n", k), ++bad;
            run(q);
        }
        const std::vector<uint16_t> got = download(whole, results), want = download(parts, results);
        if (c.norm) row_out[1][0] = download(p.shortcut_out, k), row_out[1][1] = download(p.normed_out, k);
        uint32_t differ = 0, top = 0;
        for (uint32_t i = 0; i < results; ++i) {
            differ += got[i] != want[i];
            if (bf16_to_f32(want[i]) > bf16_to_f32(want[top])) top = i;
        }
        if (differ) printf("K = %u, %u + %u rows: %u differ\n", k, c.n0, c.n1, differ), ++bad;
        for (int i = 0; i < 2; ++i)
            if (row_out[0][i] != row_out[1][i]) printf("K = %u: the normalized row differs\n", k), ++bad;
        if (c.amax) {
            const std::vector<float> value = download(top_value, grid);
            const std::vector<uint32_t> index = download(top_index, grid);
            uint32_t best = 0;
            for (uint32_t i = 1; i < grid; ++i)
                if (value[i] > value[best] || (value[i] == value[best] && index[i] < index[best])) best = i;
            if (index[best] != top) printf("K = %u, %u rows: the largest is %u, not %u\n", k, rows, index[best], top), ++bad;
        }
        hip(hipFree(d_w)), hip(hipFree(part_w));
    }
    printf("%d bad\n", bad);
    return bad != 0;
}
