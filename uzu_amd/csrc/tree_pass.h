// tree_pass.h -- what a pass over a speculated tree runs in place of the general kernels (k_tree_attention.hip).
#pragma once

#include "kernels.h"

namespace uzu {
namespace k {

constexpr uint32_t kTreeAttentionShares = 64; // shares of the keys at most, each with a partial result a column

// bf16 rows of at most 32 nodes under the trie mask alone (no window, ring or sinks), heads of 64, 128 or 256
bool attention_tree_supported(const AttentionParams& a);
// columns of partial results over all shares: partials hold head_dim floats for each, sums and maxs one
size_t attention_tree_columns(uint32_t num_heads, uint32_t gqa_factor, uint32_t nodes);
// key_rows: rows that the caches hold memory for, at least sequence_length (with dyn).
// gate (optional): SigmoidGate on the finished rows, as the kernel of that name rounds
uzu_status attention_tree(hipStream_t s, const AttentionParams& a, uint32_t key_rows, float* partials, float* sums, float* maxs, void* out, const void* gate);

} // namespace k
} // namespace uzu
