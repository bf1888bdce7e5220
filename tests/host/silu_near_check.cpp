// silu_bf16_near of uzu_math.h: for every bf16 gate and any quotient within 16 f32 ulps of the exact one the result is that of the 64-bit exponential.
#include <cmath>
#include <cstdio>
#include "../../uzu_amd/csrc/uzu_math.h"
int main() {
    unsigned long long checked = 0, bad = 0;
    for (uint32_t u = 0; u < 65536; ++u) {
        const float x = uzu::bits_to_f32(u << 16);
        const uint32_t want = uzu::f32_to_bits(uzu::activate_bf16_tab(0, x, uzu::kExp2fTab));
        const uint32_t exact = uzu::f32_to_bits((float)((double)x / (1.0 + std::exp(-(double)x))));
        for (int off = -16; off <= 16; ++off) {
            const uint32_t near = (exact & 0x7fffffffu) == 0 && off < 0 ? exact : exact + off;
            ++checked, bad += uzu::f32_to_bits(uzu::silu_bf16_near(x, uzu::bits_to_f32(near), uzu::kExp2fTab)) != want && x == x;
        }
    }
    printf("%llu checked, %llu bad\n", checked, bad);
}
