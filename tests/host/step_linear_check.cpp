// The launch of an f32-stream decode step that ends a layer and runs the projection behind it (k_step32.hip: norm_linear), called by itself: against 64 bits at widths with and without a ragged last
// piece of 512, and with an infinite weight at the end of a row, which is that row's result and nobody else's.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../uzu_amd/csrc/kernels.h"
#include "../../uzu_amd/csrc/kernels_stream32.h"
#include "../../uzu_amd/csrc/uzu_math.h"

using namespace uzu;

template <class T> static T* upload(const std::vector<T>& v) {
    T* p = nullptr;
    if (hipMalloc((void**)&p, v.size() * sizeof(T)) != hipSuccess || hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice) != hipSuccess) exit(2);
    return p;
}
template <class T> static std::vector<T> download(const T* p, size_t count) {
    std::vector<T> v(count);
    if (hipMemcpy(v.data(), p, count * sizeof(T), hipMemcpyDeviceToHost) != hipSuccess) exit(2);
    return v;
}

int main() {
    std::mt19937 rng(11);
    std::normal_distribution<float> normal;
    int bad = 0;
    for (const uint32_t d : {8u, 504u, 520u, 1024u, 1544u, 2560u, 4088u})
        for (const uint32_t n : {1u, 9u, 4112u}) {
            std::vector<float> y(d), residual(d), scales(d), next_scales(d), zero(d), out(n);
            std::vector<uint16_t> w((size_t)n * d);
            for (uint32_t i = 0; i < d; ++i) y[i] = normal(rng), residual[i] = normal(rng), scales[i] = 0.1f * normal(rng), next_scales[i] = 0.1f * normal(rng);
            for (uint16_t& x : w) x = f32_to_bf16(normal(rng));
            k::NormAddParams a{};
            a.y = upload(y), a.residual = upload(residual), a.out = upload(zero), a.scales = upload(scales), a.offset = 1.0f, a.eps = 1e-6f, a.next = upload(zero), a.next_scales = upload(next_scales);
            a.next_offset = 1.0f, a.next_eps = 1e-6f, a.rows = 1, a.d = d;
            for (const bool infinite : {false, true}) {
                if (infinite) w[(size_t)n * d - 1] = 0x7F80;
                k::LinearF32Params p{};
                p.w = upload(w), p.y = upload(out), p.rows = 1, p.n = n, p.k = d, p.ldx = d, p.ldy = n, p.batch = 1;
                float* part_value = upload(std::vector<float>(k::kNormLinearParts, NAN));
                uint32_t *part_index = upload(std::vector<uint32_t>(k::kNormLinearParts, 0)), parts = 0;
                if (k::norm_linear(nullptr, a, p, part_value, part_index, &parts) != UZU_OK) printf("%s\n", uzu_hip_last_error()), exit(2);
                if (hipDeviceSynchronize() != hipSuccess) exit(2);
                double ss = 0, ss2 = 0;
                std::vector<double> x(d);
                for (uint32_t i = 0; i < d; ++i) ss += (double)y[i] * y[i];
                for (uint32_t i = 0; i < d; ++i) x[i] = residual[i] + y[i] / std::sqrt(ss / d + 1e-6f) * (scales[i] + 1.0), ss2 += x[i] * x[i];
                for (uint32_t i = 0; i < d; ++i) x[i] = x[i] / std::sqrt(ss2 / d + 1e-6f) * (next_scales[i] + 1.0);
                const std::vector<float> got = download(p.y, n);
                uint32_t top = 0;
                for (uint32_t c = 0; c < n; ++c) {
                    if (got[c] > got[top]) top = c;
                    double want = 0, size = 0;
                    for (uint32_t i = 0; i < d; ++i) {
                        const double t = x[i] * bf16_to_f32(w[(size_t)c * d + i]);
                        want += t, size += std::fabs(t);
                    }
                    // (a lane adds at most 64 products one after the other, the norms as many; a handful of roundings each besides)
                    if (std::isinf(want) ? got[c] != (float)want : !(std::fabs(got[c] - want) <= 160 * 0x1p-24 * size)) printf("width %u, column %u of %u: %g, not %g\n", d, c, n, got[c], want), ++bad;
                }
                const std::vector<float> value = download(part_value, parts);
                const std::vector<uint32_t> index = download(part_index, parts);
                uint32_t best = 0;
                for (uint32_t i = 1; i < parts; ++i)
                    if (value[i] > value[best]) best = i;
                if (index[best] != top || value[best] != got[top]) printf("width %u, %u columns: the largest is %u, not %u\n", d, n, index[best], top), ++bad;
            }
        }
    printf("%d bad\n", bad);
    return bad != 0;
}
