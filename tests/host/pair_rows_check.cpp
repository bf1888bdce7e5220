// Products whose rows exist in pair order only (MatmulParams::a null) are refused on the host where a kernel would read plain rows: without the rows' sums, without pair rows, or for a
// product that another form takes.  And a Normalization is refused pair rows where the kernel that writes them is not the one that would run.  Nothing is launched: run without a GPU, a launch fails with another status.
#include <stdio.h>

#include "../../uzu_amd/csrc/kernels.h"

using namespace uzu::k;

int main() {
    static uint8_t memory[64] __attribute__((aligned(64))); // never read: the addresses only
    MatmulParams p{};
    p.b = memory, p.scales = memory, p.biases = memory, p.d = memory, p.pre_coef = (const float*)memory;
    p.w_dt = p.a_dt = p.d_dt = UZU_BF16, p.b_kind = UZU_MATMUL_B_SCALE_BIAS, p.bits = 4, p.group_size = 128, p.ab_scale = 1.0f;
    p.m = 512, p.n = 8192, p.k = 2048;
    int bad = 0;
    auto refused = [&](const char* what, const MatmulParams& q) {
        const uzu_status direct = gemm_q_mfma128(nullptr, q, 256, memory), dispatched = matmul(nullptr, q, 256, nullptr);
        printf("%s: %d %d\n", what, (int)direct, (int)dispatched);
        bad += direct != UZU_ERR_UNSUPPORTED || dispatched != UZU_ERR_UNSUPPORTED;
    };
    refused("no rows", p);
    p.a_pairs = (const uint16_t*)memory;
    refused("pair rows without their sums", p);
    p.pre_rowsum = (const float*)memory;
    MatmulParams other = p;
    other.group_size = 64; // the register-staged forms
    refused("another form", other);
    other = p, other.a_pairs = nullptr;
    refused("sums without rows", other);
    MatmulParams copied = p; // 512 rows of 8192 x 2048, 256 tiles; 1024 rows, 512 tiles: their copy's room only where the rows are not brought
    copied.m = 1024, copied.a = memory, copied.a_pairs = nullptr;
    MatmulParams brought = copied;
    brought.a_pairs = (const uint16_t*)memory;
    bad += gemm_q_mfma128_workspace_bytes(copied, 256) != gemm_q_mfma128_workspace_bytes(brought, 256) + (size_t)1024 * 2048 * 2;
    copied.m = brought.m = 512;
    bad += gemm_q_mfma128_workspace_bytes(copied, 256) != gemm_q_mfma128_workspace_bytes(brought, 256);
    NormParams n{};
    n.input = n.output = memory, n.scales = memory, n.pairs_out = (uint16_t*)memory, n.io_dt = UZU_BF16, n.affine_dt = UZU_F32, n.batch_size = 128, n.element_count = 1024, n.epsilon = 1e-5f;
    auto norm_refused = [&](const char* what, const NormParams& q) {
        const uzu_status status = normalization(nullptr, q);
        printf("%s: %d\n", what, (int)status);
        bad += status != UZU_ERR_UNSUPPORTED;
    };
    for (uint32_t width : {512u, 1000u, 5120u, 3072u}) {
        NormParams q = n;
        q.element_count = width;
        norm_refused("another width", q);
    }
    NormParams q = n;
    q.batch_size = 1, norm_refused("one row", q);
    q = n, q.io_dt = UZU_F32, norm_refused("f32 rows", q);
    q = n, q.affine_dt = 77, norm_refused("another scale type", q);
    q = n, q.input = memory + 4, norm_refused("input off 8 bytes", q);
    q = n, q.pairs_out = (uint16_t*)(memory + 8), norm_refused("pair rows off 16 bytes", q);
    printf("%d bad\n", bad);
    return bad;
}
