// The chunked conv1d launch, for the entry points that run it (conv1d_decode.hip
// defines it; slots are the caller's to validate).
#pragma once

#include "capi_common.h"

namespace braid {

// braid_conv1d_prefill without its slot check. pads: whether the outputs at pad
// positions (t >= seq_lens[b]) are written as 0 or left as they are.
int conv_prefill(float* conv_pool, int64_t n_slots, int C, int K, const int32_t* slot_idx, int B,
                 int T, const void* x, int x_dtype, const float* weight, const float* bias,
                 float* out, const int32_t* seq_lens, bool pads, hipStream_t stream);

}  // namespace braid
