// The large tiles' GatedActMul epilogue (gemm128_epilogue.h: SiLU from the hardware's exp2 and reciprocal, the 64-bit exponential where that could change the rounding) on the GPU, against
// activate_bf16_tab for every bf16 gate from 2^-120 to 2^120 and zero (a product's sum is + 0), on each form of the product.  A row holds its gate at k = 0; gate columns have code + 1 there and 0 elsewhere, up
// columns the scale 0 and the bias 1: the pair is (1, gate) exactly and the output SiLU(gate).
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../uzu_amd/csrc/kernels.h"
#include "../../uzu_amd/csrc/uzu_math.h"

using namespace uzu;

#define CHECK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) { printf("%s: %s\n", #x, hipGetErrorString(e_)); return 1; } } while (0)

template <class T> static T* upload(const std::vector<T>& v) {
    T* p = nullptr;
    if (hipMalloc((void**)&p, v.size() * sizeof(T)) != hipSuccess || hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice) != hipSuccess) exit(1);
    return p;
}

int main() {
    constexpr uint32_t H = 64, N = 2 * H, K = 256;
    std::vector<uint16_t> gates;
    for (uint32_t u = 0; u < 65536; ++u) {
        const float g = std::fabs(bits_to_f32(u << 16));
        if (u == 0 || (g >= std::ldexp(1.0f, -120) && g <= std::ldexp(1.0f, 120))) gates.push_back((uint16_t)u);
    }
    const uint32_t M = (uint32_t)gates.size();
    std::vector<uint16_t> rows((size_t)M * K, 0), scales(N * (K / 128)), bias(N), out((size_t)M * H);
    for (uint32_t m = 0; m < M; ++m) rows[(size_t)m * K] = gates[m];
    std::vector<uint8_t> codes((size_t)N * K / 2, 0x88);
    for (uint32_t n = 0; n < N; ++n) {
        for (uint32_t g = 0; g < K / 128; ++g) scales[n * (K / 128) + g] = n < H ? 0 : 0x3F80;
        bias[n] = n < H ? 0x3F80 : 0;
        if (n >= H) codes[(size_t)n * K / 2] = 0x89;
    }
    k::MatmulParams p{};
    p.a = upload(rows), p.b = upload(codes), p.scales = upload(scales), p.bias = upload(bias);
    uint16_t* d = upload(out);
    p.d = d, p.w_dt = p.a_dt = p.d_dt = UZU_BF16, p.b_kind = UZU_MATMUL_B_SCALE_SYMMETRIC, p.bits = 4, p.group_size = 128, p.ab_scale = 1.0f;
    p.m = M, p.n = N, p.k = K, p.act_mul = 1, p.act_type = 0;
    int bad = 0;
    for (const char* form : {"", "gemm_form=0", "gemm_form=1", "gemm_form=2"}) {
        setenv("UZU_HIP_TUNE", form, 1);
        CHECK(hipMemset(d, 0xFF, out.size() * 2));
        const char* variant = "";
        const uzu_status status = k::matmul(nullptr, p, 256, &variant);
        if (status != UZU_OK) printf("status %d: %s\n", (int)status, uzu_hip_last_error()), ++bad;
        CHECK(hipMemcpy(out.data(), d, out.size() * 2, hipMemcpyDeviceToHost));
        long wrong = 0;
        for (uint32_t m = 0; m < M; ++m) {
            const uint16_t want = (uint16_t)(f32_to_bits(activate_bf16_tab(0, bits_to_f32((uint32_t)gates[m] << 16), kExp2fTab)) >> 16);
            for (uint32_t n = 0; n < H; ++n) wrong += out[(size_t)m * H + n] != want;
        }
        printf("%s [%s]: %u gates, %ld wrong\n", variant, form, M, wrong);
        bad += wrong != 0;
    }
    printf("%d bad\n", bad);
    return bad;
}
