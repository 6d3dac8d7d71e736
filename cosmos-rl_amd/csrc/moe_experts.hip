// The experts of one MoE layer on routed tokens as one call: routing, 1x128 quantisation of the tokens, the gate_up product
// with SwiGLU, the down product and the weighted sum over each token's experts - launches only, on caller memory.
//
// Every expert's rows are padded to tiles of 128 (experts without a row get none), the tokens quantised into that layout
// (cfp8_scatter_quant_group128) and multiplied by the grouped GEMMs of the training path.  A group's rows of padding are
// zeros all the way: a walking GEMM carries a row's last products into the first step of its next tile with a scale of
// zero, so what multiplies there must be finite.  Rows past the last group are not touched, neither by the quantiser nor
// as a zero-filled output of the down product (at 8192 tokens of 2048, top 8 of 128 experts: 42 us of zeros), and the
// routing's row experts and sorted weights spare seven launches that derived them: 250 -> 230 us at 777 tokens,
// 669 -> 577 us at 8192.
#include "cfp8_common.h"

namespace cfp8 {

struct ExpertsPlan {
    int64_t rows;  // rows of the expert-grouped layout (their bound)
    size_t row_tokens, row_experts, row_map, weights, m_sizes, m_offsets, route, xq, xs, h, hs, out, bytes;
};

static ExpertsPlan experts_plan(int64_t tokens, int topk, int experts, int64_t hidden, int64_t inter) {
    ExpertsPlan p{};
    const int64_t pairs = tokens * topk;
    const int64_t touched = pairs < experts ? pairs : experts;
    p.rows = (pairs + touched * 127) / 128 * 128;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += (bytes + 255) & ~(size_t)255;
        return here;
    };
    p.row_tokens = take((size_t)p.rows * 4);
    p.row_experts = take((size_t)p.rows * 4);
    p.row_map = take((size_t)pairs * 4);
    p.weights = take((size_t)pairs * 2);
    p.m_sizes = take((size_t)experts * 4);
    p.m_offsets = take((size_t)experts * 4);
    p.route = take(cfp8_route_tokens_workspace_bytes(tokens, topk, experts));
    p.xq = take((size_t)p.rows * (size_t)hidden);
    p.xs = take((size_t)p.rows * (size_t)(hidden / 128) * 4);
    p.h = take((size_t)p.rows * (size_t)inter);
    p.hs = take((size_t)p.rows * (size_t)(inter / 128) * 4);
    p.out = take((size_t)p.rows * (size_t)hidden * 2);
    p.bytes = at;
    return p;
}

}  // namespace cfp8

extern "C" size_t cfp8_moe_experts_workspace_bytes(int64_t tokens, int topk, int experts, int64_t hidden, int64_t inter) {
    if (tokens <= 0 || topk <= 0 || experts <= 0 || hidden <= 0 || inter <= 0) return 0;
    return cfp8::experts_plan(tokens, topk, experts, hidden, inter).bytes;
}

extern "C" int cfp8_moe_experts(const void* x, int64_t ld_x, int64_t tokens, int64_t hidden, const void* indices, int index_bytes,
                                const uint8_t* token_mask, const void* weights, int weights_dtype, int topk, int experts,
                                const void* gate_up, const float* gate_up_scales, const void* down, const float* down_scales, int64_t inter,
                                void* y, int64_t ld_y, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace cfp8;
    if (tokens < 0 || hidden <= 0 || inter <= 0 || topk <= 0 || topk > 64 || experts <= 0)
        return set_error(CFP8_EINVAL, "moe_experts: tokens=%lld hidden=%lld inter=%lld topk=%d experts=%d (topk at most 64)", (long long)tokens,
                         (long long)hidden, (long long)inter, topk, experts);
    if (hidden % 128 || inter % 128) return set_error(CFP8_EINVAL, "moe_experts: hidden=%lld and inter=%lld must be multiples of 128", (long long)hidden, (long long)inter);
    if (tokens == 0) return CFP8_OK;
    if (!x || !indices || !weights || !gate_up || !gate_up_scales || !down || !down_scales || !y) return set_error(CFP8_EINVAL, "moe_experts: null pointer");
    if (!aligned16(x) || !aligned16(y) || !aligned16(gate_up) || !aligned16(down) || ld_x % 8 || ld_x < hidden || ld_y % 8 || ld_y < hidden)
        return set_error(CFP8_EINVAL, "moe_experts: misaligned pointer or bad leading dimension");
    if (tokens > 0x7FFFFFFFll / 64) return set_error(CFP8_EINVAL, "moe_experts: too many tokens");
    const ExpertsPlan p = experts_plan(tokens, topk, experts, hidden, inter);
    if (!workspace || workspace_bytes < p.bytes)
        return set_error(CFP8_EWORKSPACE, "moe_experts: workspace of %zu bytes needed, %zu given", p.bytes, workspace_bytes);
    if (reinterpret_cast<uintptr_t>(workspace) & 255u) return set_error(CFP8_EINVAL, "moe_experts: workspace must be 256-byte aligned");
    uint8_t* const ws = static_cast<uint8_t*>(workspace);
    auto i32 = [&](size_t at) { return reinterpret_cast<int32_t*>(ws + at); };
    auto f32 = [&](size_t at) { return reinterpret_cast<float*>(ws + at); };
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (int rc = cfp8_route_tokens(indices, index_bytes, token_mask, tokens, topk, experts, 128, CFP8_ROUTE_END_NOT_PADDING, p.rows,
                                   i32(p.row_tokens), i32(p.row_experts), i32(p.row_map), nullptr, weights, weights_dtype, ws + p.weights,
                                   i32(p.m_sizes), i32(p.m_offsets), ws + p.route, cfp8_route_tokens_workspace_bytes(tokens, topk, experts), stream))
        return rc;
    if (int rc = cfp8_scatter_quant_group128(x, ld_x, tokens, hidden, i32(p.row_map), topk, i32(p.row_tokens), p.rows, ws + p.xq, hidden, f32(p.xs), stream))
        return rc;
    if (int rc = cfp8_gemm_grouped_swiglu_quant(ws + p.xq, hidden, f32(p.xs), gate_up, gate_up_scales, i32(p.row_experts), ws + p.h, inter,
                                                f32(p.hs), p.rows, inter, hidden, experts, stream))
        return rc;
    if (int rc = cfp8_gemm_grouped_block128(ws + p.h, inter, f32(p.hs), down, down_scales, i32(p.row_experts), ws + p.out, hidden, CFP8_OUT_BF16,
                                            p.rows, hidden, inter, experts, stream))
        return rc;
    return cfp8_combine_rows(ws + p.out, hidden, p.rows, i32(p.row_map), ws + p.weights, CFP8_IN_BF16, tokens, topk, hidden,
                             CFP8_COMBINE_BF16_STEPS, y, ld_y, stream);
}
