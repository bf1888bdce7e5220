// tree_pass.h -- what a pass over a speculated tree runs in place of the general kernels (k_tree_attention.hip).
#pragma once

#include "kernels.h"

namespace uzu {
namespace k {

constexpr uint32_t kTreeAttentionShares = 64; // shares of the keys at most, each with a partial result a column

// bf16 rows of at most 32 nodes under the trie mask alone (no window, ring or sinks), heads of 64, 128 or 256
bool attention_tree_supported(const AttentionParams& a);
// Whether that form is the faster one in front of `keys` keys, the nodes' own among them.  two_pass: the vector form's two passes are the other choice, at whatever length; else its single
// pass.  gated: a gate follows, which the tree form applies itself.
bool attention_tree_faster(uint32_t num_heads, uint32_t gqa_factor, uint32_t head_dim, uint32_t nodes, uint32_t keys, bool two_pass, bool gated);
// columns of partial results over all shares: partials hold head_dim floats for each, sums and maxs one
size_t attention_tree_columns(uint32_t num_heads, uint32_t gqa_factor, uint32_t nodes);
// key_rows: rows that the caches hold memory for, at least sequence_length (with dyn).
// gate (optional): SigmoidGate on the finished rows, as the kernel of that name rounds
uzu_status attention_tree(hipStream_t s, const AttentionParams& a, uint32_t key_rows, float* partials, float* sums, float* maxs, void* out, const void* gate);

// ConvTreeScan, the tree's preparation and the tree-verify composite in one launch, bit-identical to delta_net_tree_prep + delta_net_tree_verify (k_deltanet_tree.hip).  Nodes in
// depth-first order (an ancestor in front of its descendants).
bool delta_net_tree_step_supported(const uint16_t* in_proj, const float* h0, uint32_t n, uint32_t kernel_size, uint32_t Hk, uint32_t Hv, uint32_t Dk, uint32_t Dv);
bool delta_net_tree_step_faster(uint32_t n, uint32_t Hv); // than the two
uzu_status delta_net_tree_step(hipStream_t s, const uint16_t* in_proj, const float* conv_w, const float* conv_b, const float* base_state, const int32_t* parents, const uint32_t* trie,
                               const float* a_log, const float* dt_bias, const float* h0, float* suffix_state, uint16_t* k_out, uint16_t* v_out, float* beta_out, float* log_decay_out,
                               uint16_t* out, uint32_t n, uint32_t kernel_size, uint32_t Hk, uint32_t Hv);

// StateAdvance of several layers along one accepted path (head_dim 128), in one launch; passed by value
struct TreeState {
    const uint16_t *k, *v;
    const float *log_decay, *beta;
    float* state;
    uint32_t Hv, Hk;
};
constexpr uint32_t kTreeStateLayers = 64; // (3.2 KB of kernel arguments)
struct TreeStates {
    TreeState layer[kTreeStateLayers];
    uint32_t accepted[kDnTreeMaxNodes], accepted_len;
};
uzu_status delta_net_states_advance(hipStream_t s, const TreeStates& t, uint32_t layers);

} // namespace k
} // namespace uzu
