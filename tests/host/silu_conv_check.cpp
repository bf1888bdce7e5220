// The quick SiLU of a prompt's convolution (csrc/silu_near.h: silu_bf16) on the device, for f32 arguments: a channel whose taps and rows are zero has its bias as its sum.  Against the rounded SiLU with
// the 64-bit exponential, the same bits: every f32 from 2^-8 to 128 in size of either sign (where the quick quotients decide, and past their border at 80), and one in 61 of the others.
// Argument "all": all 2^32.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>

#include "../../uzu_amd/csrc/kernels.h"
#include "../../uzu_amd/csrc/uzu_math.h"

using namespace uzu;

constexpr uint32_t kChannels = 1u << 22;

template <class T> static T* zeros(size_t count) {
    T* p = nullptr;
    if (hipMalloc((void**)&p, count * sizeof(T)) != hipSuccess || hipMemset(p, 0, count * sizeof(T)) != hipSuccess) exit(2);
    return p;
}

int main(int argc, char** argv) {
    const bool all = argc > 1 && !strcmp(argv[1], "all");
    const uint32_t lo = f32_to_bits(0.00390625f), hi = f32_to_bits(128.0f);
    auto next = [&](uint64_t u) { // the next bit pattern that is looked at
        const uint32_t size = (uint32_t)u & 0x7FFFFFFFu;
        return all || (size >= lo && size < hi) ? u + 1 : u + std::min<uint64_t>(61, size < lo ? lo - size : 61);
    };
    const uint16_t* rows = zeros<uint16_t>(kChannels);
    const float *weight = zeros<float>((size_t)kChannels * 4), *state = zeros<float>((size_t)kChannels * 3);
    float* bias = zeros<float>(kChannels);
    uint16_t* out = zeros<uint16_t>(kChannels);
    unsigned long long checked = 0, bad = 0;
    std::vector<float> x(kChannels);
    std::vector<uint16_t> got(kChannels);
    for (uint64_t u = 0; u < 1ull << 32;) {
        uint32_t count = 0;
        for (; count < kChannels && u < 1ull << 32; u = next(u)) x[count++] = bits_to_f32((uint32_t)u);
        std::fill(x.begin() + count, x.end(), 0.0f);
        if (hipMemcpy(bias, x.data(), (size_t)kChannels * 4, hipMemcpyHostToDevice) != hipSuccess) exit(2);
        if (k::delta_net_conv_out_of_place(nullptr, rows, weight, bias, state, out, 1, kChannels, kChannels) != UZU_OK) printf("%s\n", uzu_hip_last_error()), exit(2);
        if (hipMemcpy(got.data(), out, (size_t)kChannels * 2, hipMemcpyDeviceToHost) != hipSuccess) exit(2);
        constexpr uint32_t kThreads = 8;
        unsigned long long wrong[kThreads] = {};
        std::vector<std::thread> pool;
        for (uint32_t t = 0; t < kThreads; ++t)
            pool.emplace_back([&, t] {
                for (uint32_t i = t; i < count; i += kThreads) {
                    const float sum = x[i] + 0.0f; // (the convolution's sum of a bias of -0 is 0)
                    const uint16_t want = f32_to_bf16(silu_f32_tab(sum, kExp2fTab));
                    if (sum != sum ? bf16_to_f32(got[i]) == bf16_to_f32(got[i]) : got[i] != want) {
                        if (!wrong[t]++) printf("%a: %04x, not %04x\n", sum, got[i], want);
                    }
                }
            });
        for (std::thread& t : pool) t.join();
        for (unsigned long long w : wrong) bad += w;
        checked += count;
        if (all && u % (1ull << 28) < kChannels) printf("at %llx\n", (unsigned long long)u), fflush(stdout);
    }
    printf("%llu arguments checked\n%llu bad\n", checked, bad);
    return bad != 0;
}
