// Routing of a MoE layer's tokens together with their 1x128 quantisation, which does not depend on it.
#pragma once

#include "quant_group.h"

namespace cfp8 {

// cfp8_route_tokens; with `tokens_q` its launches quantise those rows as well
int route_and_quantise(const void* indices, int index_bytes, const uint8_t* token_mask, int64_t tokens, int topk, int experts, int64_t alignment, int flags,
                       int64_t capacity, int32_t* row_tokens, int32_t* row_experts, int32_t* row_map, int64_t* slot_order, const void* weights,
                       int weights_dtype, void* sorted_weights, int32_t* m_sizes, int32_t* m_offsets, void* workspace, size_t workspace_bytes,
                       const GroupRows* tokens_q, hipStream_t st);

}  // namespace cfp8
