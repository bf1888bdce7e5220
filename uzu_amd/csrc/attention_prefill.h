// attention_prefill.h -- attention_prefill_mfma (k_attention_mfma.hip) for a caller that knows more than its parameters say.
#pragma once

#include "kernels.h"

namespace uzu {
namespace k {

// `prefix`: the cached keys, where AttentionParams::dyn has their number on the device; how the keys are shared out rests on it, and with that the order of the f32 sums
uzu_status attention_prefill_mfma_behind(hipStream_t s, const AttentionParams& p, uint32_t prefix, void* out, const void* gate, uint32_t* gate_done);
// the shares of the keys that its plan gives a query at most; 1: no shares and no merge
uint32_t attention_prefill_mfma_shares(const AttentionParams& p, uint32_t prefix, bool gated);

} // namespace k
} // namespace uzu
