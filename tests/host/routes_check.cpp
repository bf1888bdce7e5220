// Which kernel a call goes to, where two are right and one is faster: the rules of the library's dispatch at the sizes that their comments quote measurements for.  Host arithmetic alone.
#include <cstdio>
#include <vector>

#include "../../uzu_amd/csrc/attention_prefill.h"
#include "../../uzu_amd/csrc/kernels.h"
#include "../../uzu_amd/csrc/kernels_decode.h"
#include "../../uzu_amd/csrc/kernels_stream32.h"
#include "../../uzu_amd/csrc/tree_pass.h"

using namespace uzu::k;

namespace uzu { namespace k { bool window_attention_f32_supported(const WindowAttentionParams& p); } } // (between k_window_attention.hip and k_window_attention_f32.hip)

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
                          {24, 8, 64, 4, 180, false, false, false}, {32, 8, 128, 20, 70, false, false, false}, {32, 8, 128, 13, 110, false, false, true}, {12, 4, 128, 4, 1700, true, false, false}, {40, 8, 128, 16, 120, false, false, false}, {16, 2, 128, 1, 10, false, false, true}, {8, 2, 256, 13, 300, false, true, true},
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
                            {8, 2, 256, 517, 0, false, 4, 12}, {8, 2, 256, 517, 0, true, 4, 12}, {8, 2, 256, 2043, 0, true, 2, 4}, {8, 2, 256, 3000, 0, false, 2, 5}, {32, 8, 128, 1021, 0, false, 1, 1}, {8, 2, 256, 831, 0, false, 6, 12},
                            {8, 2, 256, 347, 600, false, 6, 12}, {8, 2, 256, 654, 0, true, 4, 12}, {24, 4, 256, 90, 600, true, 6, 12}, {16, 4, 128, 1025, 4500, false, 3, 5}, {32, 8, 128, 90, 600, false, 1, 6}}) {
        AttentionParams a{};
        a.dt = UZU_BF16, a.head_dim = t.head_dim, a.gqa_factor = t.heads / t.kv_heads, a.num_heads = t.heads, a.suffix_length = t.rows, a.sequence_length = t.rows + t.prefix, a.is_causal = 1;
        const uint32_t shares = attention_prefill_mfma_shares(a, t.prefix, t.gated);
        if (shares < t.least || shares > t.most) printf("prompt attention, %u heads on %u of %u, %u rows behind %u keys: %u shares\n", t.heads, t.kv_heads, t.head_dim, t.rows, t.prefix, shares), ++bad;
    }
    struct Window {
        uint32_t rows, heads, kv_heads, dim, window, keys;
        bool want;
    };
    for (const bool step : {true, false})
        for (const Window& t : step ? std::vector<Window>{{8, 16, 4, 128, 1024, 0, true}, {48, 32, 8, 128, 0, 4000, true}, {2, 64, 8, 64, 1024, 1300, true}, {8, 64, 8, 64, 1024, 1300, false}, {12, 64, 8, 64, 0, 300, true},
                                                          {12, 64, 8, 64, 0, 3900, false}, {6, 64, 8, 64, 1024, 1300, false}, {24, 64, 8, 64, 3000, 150, true}, {4, 40, 8, 128, 512, 450, true}, {12, 40, 8, 128, 1024, 1300, true},
                                                          {4, 24, 2, 128, 1024, 1300, true}, {32, 24, 2, 128, 512, 450, false}, {12, 24, 2, 128, 0, 300, true}, {48, 24, 2, 128, 3000, 150, true},
                                                          {48, 24, 2, 128, 0, 3900, false}, {32, 48, 3, 64, 3000, 150, true}, {32, 48, 3, 64, 3000, 1999, false}, {1, 16, 1, 128, 0, 0, true}}
                                    : std::vector<Window>{{300, 8, 2, 128, 0, 0, true}, {16, 8, 2, 128, 0, 0, true}, {16, 8, 2, 128, 64, 0, false}, {64, 16, 4, 128, 64, 0, false}, {200, 8, 2, 128, 64, 0, true},
                                                          {32, 8, 2, 128, 128, 0, false}, {16, 8, 2, 128, 192, 0, true}, {300, 8, 2, 128, 1024, 0, true}}) {
            WindowAttentionParams p{};
            p.rows = t.rows, p.nseq = step ? t.rows : 1, p.heads = t.heads, p.kv_heads = t.kv_heads, p.dim = p.vdim = t.dim, p.ldq = t.heads * t.dim, p.window = t.window, p.keys = t.keys, p.one_row = step, p.cache_bf16 = step;
            if (step) p.tiles = p.tiles32 = t.rows, window_attention_split_keys(p, t.window ? t.window : 4096, 256);
            char what[160];
            snprintf(what, sizeof what, "%s attention, %u rows of %u heads on %u of %u, window %u, %u keys", step ? "step" : "f32 prompt", t.rows, t.heads, t.kv_heads, t.dim, t.window, t.keys);
            expect(step ? p.split_items == 0 : window_attention_f32_supported(p), t.want, what);
        }
    for (const uint32_t outputs : {8u, 32u, 64u})
        for (const uint32_t d : {256u, 1024u, 2048u}) {
            RouteGroupsParams p{};
            p.outputs = outputs, p.d = d, p.rows = 8, p.top = 2;
            char what[100];
            snprintf(what, sizeof what, "norm and routing of %u outputs, rows of %u", outputs, d);
            expect(norm_route_faster(p), outputs <= 32 || d == 2048, what);
        }
    for (const uint32_t heads : {4u, 32u, 48u, 64u, 72u})
        for (const uint32_t nodes : {1u, 10u, 13u, 16u, 17u, 28u, 32u}) {
            char what[100];
            snprintf(what, sizeof what, "a tree's DeltaNet layer in one launch, %u heads, %u nodes", heads, nodes);
            expect(delta_net_tree_step_faster(nodes, heads), heads <= 32 || (heads == 72 ? nodes >= 13 : nodes == 17 || nodes == 28), what);
        }
    struct Large {
        uint32_t n, k, act_mul;
        bool want;
    };
    for (const Large& t : {Large{2048, 4096, 0, true}, {2046, 4096, 0, false}, {2048, 4096, 1, false}, {2144, 4096, 1, true}, {2048, 8192, 1, false}, {2560, 8192, 1, true}, {6144, 2048, 1, false}, {6400, 2048, 1, true},
                           {4096, 2048, 0, true}, {28672, 4096, 1, true}, {28672, 4064, 0, false}}) {
        DecGemvParams p{};
        p.n[0] = t.n, p.k = t.k, p.bits = 8, p.b_kind = UZU_MATMUL_B_SCALE_BIAS, p.group_size = 32, p.act_mul = t.act_mul;
        char what[100];
        snprintf(what, sizeof what, "the stream of an int8 matrix of %u rows of %u%s", t.n, t.k, t.act_mul ? ", gated" : "");
        expect(gemv_large_wanted(p, 256), t.want, what);
    }
    { // a decode step's joined launches: refused where a workgroup would write what another may still read
        const auto at = [](size_t floats) { return (float*)(0x10000000 + 4 * floats); }; // (never read)
        const uint32_t d = 1024;
        for (const size_t written : {0u, 1020u, 1024u, 2044u, 2048u, 4096u}) // the sublayer's result lies at 0, the stream's row at 1024
            for (const int which : {0, 1, 2}) {
                NormAddParams n{};
                n.y = at(0), n.residual = at(d), n.out = at(which == 0 ? written : 8192), n.next = at(which == 1 ? written : 16384), n.scales = n.next_scales = at(32768), n.rows = 1, n.d = d;
                LinearF32Params p{};
                p.w = (const uint16_t*)at(65536), p.y = at(which == 2 ? written : 131072), p.rows = p.batch = 1, p.n = 4112, p.k = d;
                RouteGroupsParams r{};
                r.router = (const uint16_t*)at(65536), r.ids = (int32_t*)at(262144), r.weights = at(262208), r.rows = 1, r.d = d, r.outputs = 8, r.top = 2, r.groups = r.keep = 1;
                char what[100];
                snprintf(what, sizeof what, "a step's launch whose %s lies %zu floats behind the sublayer's result", which == 0 ? "new row" : which == 1 ? "norm" : "product", written);
                expect(norm_linear_supported(n, p), written >= 2048, what);
                if (which < 2) expect(norm_route_gate_up_supported(n, r, (const uint16_t*)at(524288), 1024, ExpertAct()), written >= 2048, what);
            }
    }
    printf("%d bad\n", bad);
    return bad != 0;
}
