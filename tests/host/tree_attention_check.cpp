// The tree form of attention (k_tree_attention.hip) on the GPU, called by itself at its edges, whatever the dispatch would choose: against the vector form's two passes, within two bf16 ulps or
// 2e-3 (both take f32 sums of the same exact products, in other orders), and with NaN in the caches' rows behind the last key, which it loads: the same bits as with zeros there.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../uzu_amd/csrc/kernels.h"
#include "../../uzu_amd/csrc/tree_pass.h"
#include "../../uzu_amd/csrc/uzu_math.h"

using namespace uzu;

template <class T> static T* upload(const std::vector<T>& v) {
    T* p = nullptr;
    if (hipMalloc((void**)&p, v.size() * sizeof(T)) != hipSuccess || hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice) != hipSuccess) exit(2);
    return p;
}
static void need(uzu_status st) {
    if (st != UZU_OK) printf("status %d: %s\n", (int)st, uzu_hip_last_error()), exit(2);
}

int main() {
    struct Case {
        uint32_t nodes, heads, kv_heads, head_dim, prefix;
    };
    std::mt19937 rng(7);
    std::normal_distribution<float> normal;
    int bad = 0;
    // (a column tile that is full, one over and nearly empty, groups of columns past 64, a first tile of keys that is the tree's own, shares with none, one and several tiles)
    for (const Case& c : {Case{1, 4, 4, 64, 0}, {2, 8, 2, 128, 1}, {13, 8, 2, 256, 1023}, {16, 16, 4, 64, 31}, {17, 14, 2, 64, 96}, {31, 6, 3, 256, 32}, {32, 8, 1, 128, 2100}, {5, 8, 8, 128, 700}}) {
        const uint32_t n = c.nodes, length = c.prefix + n, rows = length + 40, hd = c.head_dim, gqa = c.heads / c.kv_heads;
        std::vector<uint32_t> trie(3 * n), path;
        for (uint32_t i = 0; i < n; ++i) { // depth-first: deeper, or back up a few nodes first
            while (path.size() > 1 && rng() % 9 < 4) path.pop_back();
            trie[3 * i] = i, trie[3 * i + 2] = (uint32_t)path.size();
            path.push_back(i);
            for (uint32_t p : path) trie[3 * p + 1] = i;
        }
        auto random = [&](size_t count) {
            std::vector<uint16_t> v(count);
            for (uint16_t& x : v) x = f32_to_bf16(normal(rng));
            return v;
        };
        std::vector<uint16_t> q = random((size_t)c.heads * n * hd), k = random((size_t)rows * c.kv_heads * hd), v = random((size_t)rows * c.kv_heads * hd), out[3];
        k::AttentionParams a{};
        a.queries = upload(q), a.trie = upload(trie), a.dt = UZU_BF16, a.head_dim = hd, a.gqa_factor = gqa, a.sequence_length = length, a.k_head_stride = a.v_head_stride = hd;
        a.k_seq_stride = a.v_seq_stride = c.kv_heads * hd, a.scale = 1.0f / std::sqrt((float)hd), a.num_heads = c.heads, a.suffix_length = n, a.is_causal = 1;
        const size_t columns = std::max(k::attention_tree_columns(c.heads, gqa, n), (size_t)n * c.heads * 32);
        float* partials = upload(std::vector<float>(columns * hd)); // NaN there too: what a share did not write is not read
        float *sums = upload(std::vector<float>(columns)), *maxs = upload(std::vector<float>(columns));
        uint16_t* d_out = upload(std::vector<uint16_t>(q.size()));
        for (int form = 0; form < 3; ++form) { // two passes; the tree form, zeros behind; NaNs behind
            std::fill(k.begin() + (size_t)length * c.kv_heads * hd, k.end(), form == 2 ? 0x7FC0 : 0);
            std::fill(v.begin() + (size_t)length * c.kv_heads * hd, v.end(), form == 2 ? 0x7FC0 : 0);
            a.keys = upload(k), a.values = upload(v);
            if (hipMemset(partials, 0xFF, columns * hd * 4) != hipSuccess || hipMemset(d_out, 0xFF, q.size() * 2) != hipSuccess) return 2;
            if (!k::attention_tree_supported(a)) return 2;
            if (form == 0) need(k::attention_two_pass1(nullptr, a, partials, sums, maxs)), need(k::attention_two_pass2(nullptr, partials, sums, maxs, d_out, UZU_BF16, hd, c.heads, n));
            else need(k::attention_tree(nullptr, a, rows, partials, sums, maxs, d_out, nullptr));
            out[form].resize(q.size());
            if (hipMemcpy(out[form].data(), d_out, q.size() * 2, hipMemcpyDeviceToHost) != hipSuccess) return 2;
        }
        long far = 0, other = 0;
        for (size_t i = 0; i < q.size(); ++i) {
            const float x = bits_to_f32((uint32_t)out[0][i] << 16), y = bits_to_f32((uint32_t)out[1][i] << 16), d = std::fabs(x - y);
            far += !(d <= 2e-3f || d <= 2.0f * std::ldexp(1.0f, std::ilogb(std::max(std::fabs(x), std::fabs(y))) - 7));
            other += out[1][i] != out[2][i];
        }
        printf("%2u nodes, %2u heads on %u of %3u, behind %4u keys: %ld far, %ld changed by what is behind the last key\n", n, c.heads, c.kv_heads, hd, c.prefix, far, other);
        bad += far != 0 || other != 0;
    }
    printf("%d bad\n", bad);
    return bad != 0;
}
