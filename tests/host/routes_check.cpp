// Which kernel a call goes to, where two are right and one is faster: the rules of the library's dispatch at the sizes that their comments quote measurements for.  Host arithmetic alone.
#include <cstdio>

#include "../../uzu_amd/csrc/attention_prefill.h"
#include "../../uzu_amd/csrc/kernels.h"
#include "../../uzu_amd/csrc/tree_pass.h"

using namespace uzu::k;

static int bad = 0;
static void expect(bool got, bool want, const char* what) {
    if (got != want) printf("%s: %s\n", what, got ? "taken" : "not taken"), ++bad;
}

int main() {
    struct Tree {
        uint32_t heads, kv_heads, head_dim, nodes, context;
        bool two_pass, gated, want;
    };
    for (const Tree& t : {Tree{16, 16, 128, 13, 80, false, false, false}, {16, 16, 128, 13, 600, false, false, true}, {8, 8, 64, 13, 250, false, false, false}, {8, 8, 64, 13, 600, false, false, true},
                          {8, 8, 256, 2, 80, false, false, false}, {8, 8, 256, 2, 250, false, false, true}, {32, 8, 128, 1, 30, false, false, false}, {32, 8, 128, 1, 250, false, false, true},
                          {24, 8, 64, 4, 180, false, false, false}, {40, 8, 128, 16, 120, false, false, false}, {16, 2, 128, 1, 10, false, false, true}, {8, 2, 256, 13, 300, false, true, true},
                          {16, 16, 128, 4, 1500, true, false, false}, {16, 16, 128, 8, 1500, true, false, true}, {32, 8, 128, 1, 4000, true, false, false}, {32, 8, 128, 3, 1500, true, false, true},
                          {8, 4, 256, 6, 1500, true, false, false}, {8, 4, 256, 8, 4000, true, false, true}, {8, 2, 256, 2, 1500, true, true, true}, {8, 2, 256, 13, 1500, true, true, true},
                          {2, 2, 128, 16, 8000, true, false, false}, {32, 32, 128, 2, 8000, true, false, false}, {32, 32, 128, 6, 8000, true, false, true}, {64, 8, 64, 1, 1100, true, false, true}}) {
        char what[160];
        snprintf(what, sizeof what, "tree attention, %u heads on %u of %u, %u nodes behind %u keys", t.heads, t.kv_heads, t.head_dim, t.nodes, t.context);
        expect(attention_tree_faster(t.heads, t.heads / t.kv_heads, t.head_dim, t.nodes, t.context + t.nodes, t.two_pass, t.gated), t.want, what);
    }
    struct Prompt {
        uint32_t heads, kv_heads, head_dim, rows, prefix;
        bool gated;
        uint32_t least, most; // shares of the keys
    };
    for (const Prompt& t : {Prompt{32, 8, 128, 100, 0, false, 1, 1}, {32, 8, 128, 257, 0, false, 1, 1}, {32, 8, 128, 517, 0, false, 1, 1}, {16, 4, 128, 257, 0, false, 1, 1}, {24, 8, 64, 517, 0, false, 1, 1},
                            {40, 8, 128, 130, 0, false, 1, 1}, {8, 2, 256, 100, 0, false, 1, 1}, {32, 8, 128, 64, 1000, false, 4, 12}, {16, 4, 128, 517, 2000, false, 2, 12}, {4, 4, 64, 1024, 3000, false, 4, 12},
                            {8, 2, 256, 517, 0, false, 4, 12}, {8, 2, 256, 517, 0, true, 4, 12}, {8, 2, 256, 2043, 0, true, 2, 4}, {8, 2, 256, 3000, 0, false, 2, 2}, {32, 8, 128, 1021, 0, false, 1, 1}}) {
        AttentionParams a{};
        a.dt = UZU_BF16, a.head_dim = t.head_dim, a.gqa_factor = t.heads / t.kv_heads, a.num_heads = t.heads, a.suffix_length = t.rows, a.sequence_length = t.rows + t.prefix, a.is_causal = 1;
        const uint32_t shares = attention_prefill_mfma_shares(a, t.prefix, t.gated);
        if (shares < t.least || shares > t.most) printf("prompt attention, %u heads on %u of %u, %u rows behind %u keys: %u shares\n", t.heads, t.kv_heads, t.head_dim, t.rows, t.prefix, shares), ++bad;
    }
    printf("%d bad\n", bad);
    return bad != 0;
}
