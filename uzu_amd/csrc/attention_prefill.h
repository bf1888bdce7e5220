// attention_prefill.h -- attention_prefill_mfma (k_attention_mfma.hip) for a caller that knows more than its parameters say.
#pragma once

#include "kernels.h"

namespace uzu {
namespace k {

// `prefix`: the cached keys, where AttentionParams::dyn has their number on the device; how the keys are shared out rests on it, no result does
uzu_status attention_prefill_mfma_behind(hipStream_t s, const AttentionParams& p, uint32_t prefix, void* out, const void* gate, uint32_t* gate_done);

} // namespace k
} // namespace uzu
