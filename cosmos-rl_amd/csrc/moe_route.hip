// Token routing for the grouped experts: from the top-k expert indices of every token to the expert-grouped row
// layout, in one launch (few pairs) or two.
//
// The (token, slot) pairs are numbered t * topk + s and sorted stably by expert: groups in expert order, pairs
// ascending inside a group, every group padded to a multiple of `alignment` rows.  A stable sort by a key of at most
// 1024 values is a counting sort; what it needs is every pair's rank among the pairs of its expert in front of it:
//   * inside a wave by comparing keys with ballots, one per bit of the key (the lanes that agree with this one in every
//     bit are the pairs of the same expert; the rank is the number of those below it);
//   * across the 16 waves of a workgroup by a table of counts in LDS ([wave][expert]) turned into prefix sums;
//   * across workgroups by the histograms of the workgroups in front of this one, which a first launch has written.
//
// What bounds it: nothing but latency - 65536 pairs are half a megabyte of indices and outputs of the same size.  So no load
// waits for another: a thread's own pair, its weight, its token's other slots and the mask are requested together, before the
// histograms are, and the mask decides afterwards.  The tokens' 1x128 quantisation, which needs nothing of the routing, runs in workgroups
// behind its own instead of in a launch behind it.  Routing and quantising, top 8 of 128 experts of 2048, in a kernel trace: 16 tokens 7.8 + 4.8 us in two
// launches, 6.5 in one; 777 tokens 4.7 + 8.8 + 5.1 in three, 4.8 + 8.4 in two; 8192 tokens 4.7 + 11.8 + 11.9, 4.9 + 15.8.
// The same layout built from library calls (a stable argsort, a scatter-add for the counts, a sort along the slots,
// gathers, comparisons and fills, each over 10^2 .. 10^5 elements) is some thirty launches of 2 .. 45 us each:
// 230-250 us at every size from 16 to 8192 tokens.
#include "moe_route.h"

namespace cfp8 {

constexpr int kRouteThreads = 1024, kRouteWaves = kRouteThreads / 64;
constexpr int kRouteMaxExperts = 1024;
// Pairs up to which one workgroup does it all (its histogram included): one round of the placing loop, 8 us.  2048 pairs
// take 14 us that way and 12 us in two launches.
constexpr int kRouteOneLaunchPairs = 1024;
constexpr int kRouteMaxBlocks = 128;

struct RouteArgs {
    const void* indices;      // [tokens, topk] int32 or int64
    const uint8_t* mask;      // [tokens] or null: tokens with 0 go to no expert
    const void* weights;      // [tokens, topk] bf16 or fp32, or null
    int32_t* hist;            // [blocks, experts], two launches only
    int32_t* row_tokens;      // [capacity]
    int32_t* row_experts;     // [capacity] or null
    int32_t* row_map;         // [tokens, topk]
    int64_t* slot_order;      // [tokens, topk] or null
    uint16_t* sorted_weights; // [tokens, topk] bf16 or null
    int32_t* m_sizes;         // [experts]
    int32_t* m_offsets;       // [experts]
    int64_t pairs, capacity, alignment, chunk;
    int topk, experts, bits;
    int idx64, w32, flags;
    int blocks;               // workgroups of the routing; those behind them quantise
};

__device__ __forceinline__ bool route_masked(const RouteArgs& p, int64_t token) { return p.mask && !p.mask[token]; }
// expert of a pair whose token is not masked; `experts` for an index that no expert has
__device__ __forceinline__ int route_expert(const RouteArgs& p, int64_t pair) {
    const int64_t e = p.idx64 ? static_cast<const int64_t*>(p.indices)[pair] : (int64_t) static_cast<const int32_t*>(p.indices)[pair];
    return e >= 0 && e < p.experts ? (int)e : p.experts;
}

// A pair as its thread places it.
struct RoutePair {
    int expert, token, place;  // its expert, its place among its token's slots: ascending by expert, slots of one expert in their order
    u32 pair;
    uint16_t weight;
};
__device__ __forceinline__ RoutePair route_pair(const RouteArgs& p, u32 pair, bool have) {
    RoutePair r{p.experts, 0, 0, pair, 0};
    if (!have) return r;
    r.token = (int)(pair / (u32)p.topk);
    const int slot0 = r.token * p.topk, s = (int)pair - slot0;
    // (no load waits for another: the mask decides about what they bring)
    const int expert = route_expert(p, pair);
    if (p.sorted_weights)
        r.weight = p.w32 ? (uint16_t)(pack_bf16x2(static_cast<const float*>(p.weights)[pair], 0.f) & 0xFFFFu) : static_cast<const uint16_t*>(p.weights)[pair];
    const bool masked = route_masked(p, r.token);
#pragma unroll 8
    for (int k = 0; k < p.topk; ++k) {
        const int o = route_expert(p, slot0 + k);
        r.place += o < expert || (o == expert && k < s);
    }
    if (masked) r.place = s;
    else r.expert = expert;
    return r;
}

// The workgroups behind the routing's own quantise the tokens, which it does not read.
// (Four groups a thread: one instead changed nothing from 256 to 131072 groups, whose casts run while the routing waits.)
constexpr u32 kRouteQuantGroups = kRouteThreads / 16 * 4;  // a workgroup's
__device__ __forceinline__ void route_quantise(const GroupRows& q, u32 block) {
    group128_some<CFP8_GROUP_MODE_DIV, 4>(q, block * kRouteQuantGroups + (threadIdx.x >> 4) * 4u);
}

__global__ __launch_bounds__(kRouteThreads) void route_count_kernel(const RouteArgs p) {
    __shared__ int hist[kRouteMaxExperts];
    const int t = threadIdx.x;
    const int64_t first = (int64_t)blockIdx.x * p.chunk;
    const int64_t last = first + p.chunk < p.pairs ? first + p.chunk : p.pairs;
    for (int e = t; e < p.experts; e += kRouteThreads) hist[e] = 0;
    __syncthreads();
    for (int64_t i = first + t; i < last; i += kRouteThreads) {
        const int e = route_expert(p, i);
        if (!route_masked(p, (u32)i / (u32)p.topk) && e < p.experts) atomicAdd(&hist[e], 1);
    }
    __syncthreads();
    for (int e = t; e < p.experts; e += kRouteThreads) p.hist[(int64_t)blockIdx.x * p.experts + e] = hist[e];
}

template <bool ONE>
__global__ __launch_bounds__(kRouteThreads) void route_place_kernel(const RouteArgs p, const GroupRows q) {
    __shared__ int total[kRouteMaxExperts];   // pairs of every expert
    __shared__ int base[kRouteMaxExperts];    // next row of every expert for this workgroup
    __shared__ int ends[kRouteMaxExperts];    // inclusive cumulative group ends
    __shared__ int wave_sum[kRouteWaves];
    extern __shared__ uint16_t counts[];      // [wave][experts rounded up to even]
    if ((int)blockIdx.x >= p.blocks) return route_quantise(q, blockIdx.x - p.blocks);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int E = p.experts, EP = (E + 1) & ~1;
    const int64_t first = (int64_t)blockIdx.x * p.chunk;
    const int64_t last = first + p.chunk < p.pairs ? first + p.chunk : p.pairs;
    // (the first round's pairs are on their way while the histograms are)
    RoutePair r = route_pair(p, (u32)(first + t), first + t < last);
    for (int e = t; e < E; e += kRouteThreads) total[e] = 0, base[e] = 0;
    __syncthreads();
    if (ONE) {
        if (r.expert < E) atomicAdd(&total[r.expert], 1);
    } else {
        // thread (part, expert): an expert's counts are added up by as many threads as there are, a load a workgroup each
        const int parts = kRouteThreads / E, part = t / E, e = t - part * E;
        if (part < parts) {
            int sum = 0, before = 0;
#pragma unroll 8
            for (int b = part; b < p.blocks; b += parts) {
                const int c = p.hist[b * E + e];
                sum += c;
                before += b < (int)blockIdx.x ? c : 0;
            }
            if (sum) atomicAdd(&total[e], sum);
            if (before) atomicAdd(&base[e], before);
        }
    }
    __syncthreads();
    // padded group sizes and their inclusive prefix sum, one expert per thread
    {
        u32 size = 0;
        if (t < E) {
            size = (u32)total[t];
            const u32 unit = (u32)p.alignment;
            if ((p.flags & CFP8_ROUTE_KEEP_EMPTY) && size < unit) size = unit;
            size = (size + unit - 1) / unit * unit;
        }
        int run = (int)size;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int v = __shfl_up(run, off);
            if (lane >= off) run += v;
        }
        if (lane == 63) wave_sum[wave] = run;
        __syncthreads();
        if (wave * 64 < E)
            for (int w = 0; w < wave; ++w) run += wave_sum[w];
        if (t < E) {
            ends[t] = run;
            base[t] += run - (int)size;
            if (blockIdx.x == 0) {
                p.m_sizes[t] = (int)size;
                p.m_offsets[t] = run;
            }
        }
        __syncthreads();
    }
    for (int64_t i0 = first; i0 < last; i0 += kRouteThreads) {
        for (int c = t; c < kRouteWaves * EP / 2; c += kRouteThreads) reinterpret_cast<u32*>(counts)[c] = 0;
        if (i0 != first) r = route_pair(p, (u32)(i0 + t), i0 + t < last);
        const int e = r.expert;
        uint64_t same = __ballot(e < E);
        for (int b = 0; b < p.bits; ++b) {
            const uint64_t m = __ballot((e >> b) & 1);
            same &= ((e >> b) & 1) ? m : ~m;
        }
        const int rank = __popcll(same & ((1ull << lane) - 1));
        __syncthreads();
        if (e < E && rank == 0) counts[wave * EP + e] = (uint16_t)__popcll(same);
        __syncthreads();
        int added = 0;
        if (t < E) {
#pragma unroll
            for (int w = 0; w < kRouteWaves; ++w) {
                const int c = counts[w * EP + t];
                counts[w * EP + t] = (uint16_t)added;
                added += c;
            }
        }
        __syncthreads();
        int row = -1;
        if (e < E) row = base[e] + counts[wave * EP + e] + rank;
        if (row >= p.capacity) row = -1;
        if (row >= 0) {
            p.row_tokens[row] = r.token;
            if (p.row_experts) p.row_experts[row] = e;
        }
        if (i0 + t < last) {
            const int64_t slot0 = (int64_t)r.token * p.topk;
            p.row_map[slot0 + r.place] = row;
            if (p.slot_order) p.slot_order[slot0 + r.place] = (int64_t)r.pair - slot0;
            if (p.sorted_weights) p.sorted_weights[slot0 + r.place] = r.weight;
        }
        __syncthreads();
        if (t < E) base[t] += added;
        // (the next round's first barrier orders this against its readers)
    }
    // padding: the rows behind every group's last pair, and the rows past the last group
    // (a wave per expert: the whole workgroup on one expert after the other took 25 us for 128 of them)
    for (int e = blockIdx.x * kRouteWaves + wave; e < E; e += p.blocks * kRouteWaves) {
        const int end = ends[e], start = e ? ends[e - 1] : 0;
        for (int64_t row = start + (int64_t)total[e] + lane; row < end && row < p.capacity; row += 64) {
            p.row_tokens[row] = -1;
            if (p.row_experts) p.row_experts[row] = e;
        }
    }
    for (int64_t row = (int64_t)ends[E - 1] + (int64_t)blockIdx.x * kRouteThreads + t; row < p.capacity; row += (int64_t)p.blocks * kRouteThreads) {
        p.row_tokens[row] = (p.flags & CFP8_ROUTE_END_NOT_PADDING) ? 0x7FFFFFFF : -1;
        if (p.row_experts) p.row_experts[row] = -1;
    }
}

static int64_t route_blocks(int64_t pairs) {
    if (pairs <= kRouteOneLaunchPairs) return 1;
    const int64_t rounds = (pairs + (int64_t)kRouteThreads * kRouteMaxBlocks - 1) / ((int64_t)kRouteThreads * kRouteMaxBlocks);
    return (pairs + rounds * kRouteThreads - 1) / (rounds * kRouteThreads);
}

}  // namespace cfp8

extern "C" size_t cfp8_route_tokens_workspace_bytes(int64_t tokens, int topk, int experts) {
    if (tokens <= 0 || topk <= 0 || experts <= 0) return 0;
    const int64_t blocks = cfp8::route_blocks(tokens * topk);
    return blocks == 1 ? 0 : (size_t)blocks * (size_t)experts * 4;
}

namespace cfp8 {

int route_and_quantise(const void* indices, int index_bytes, const uint8_t* token_mask, int64_t tokens, int topk, int experts,
                                 int64_t alignment, int flags, int64_t capacity, int32_t* row_tokens, int32_t* row_experts,
                                 int32_t* row_map, int64_t* slot_order, const void* weights, int weights_dtype, void* sorted_weights,
                                 int32_t* m_sizes, int32_t* m_offsets, void* workspace, size_t workspace_bytes, const GroupRows* tokens_q, hipStream_t st) {
    if (tokens < 0 || topk <= 0 || experts <= 0 || experts > kRouteMaxExperts || alignment <= 0 || capacity < 0)
        return set_error(CFP8_EINVAL, "route_tokens: tokens=%lld topk=%d experts=%d alignment=%lld capacity=%lld (1 .. %d experts)",
                         (long long)tokens, topk, experts, (long long)alignment, (long long)capacity, kRouteMaxExperts);
    if (tokens > 0x7FFFFFFFll / topk || capacity > 0x7FFFFFFFll || alignment > (1 << 20) || tokens * topk + experts * alignment > 0x7FFFFFFFll)
        return set_error(CFP8_EINVAL, "route_tokens: more than 2^31 rows");
    if (index_bytes != 4 && index_bytes != 8) return set_error(CFP8_EINVAL, "route_tokens: indices must be int32 or int64");
    if (sorted_weights && weights_dtype != CFP8_IN_BF16 && weights_dtype != CFP8_IN_F32)
        return set_error(CFP8_EINVAL, "route_tokens: weights must be bf16 or fp32");
    if (!m_sizes || !m_offsets || (tokens > 0 && (!indices || !row_map)) || (capacity > 0 && !row_tokens) || (tokens > 0 && sorted_weights && !weights))
        return set_error(CFP8_EINVAL, "route_tokens: null pointer");
    const size_t need = cfp8_route_tokens_workspace_bytes(tokens, topk, experts);
    if (need && (!workspace || workspace_bytes < need))
        return set_error(CFP8_EWORKSPACE, "route_tokens: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
    if (int rc = check_device()) return rc;
    RouteArgs p{};
    p.indices = indices;
    p.mask = token_mask;
    p.weights = weights;
    p.hist = static_cast<int32_t*>(workspace);
    p.row_tokens = row_tokens;
    p.row_experts = row_experts;
    p.row_map = row_map;
    p.slot_order = slot_order;
    p.sorted_weights = static_cast<uint16_t*>(sorted_weights);
    p.m_sizes = m_sizes;
    p.m_offsets = m_offsets;
    p.pairs = tokens * topk;
    p.capacity = capacity;
    p.alignment = alignment;
    p.topk = topk;
    p.experts = experts;
    p.bits = experts > 1 ? 32 - __builtin_clz((unsigned)experts - 1) : 0;
    p.idx64 = index_bytes == 8;
    p.w32 = weights_dtype == CFP8_IN_F32;
    p.flags = flags;
    const int64_t blocks = route_blocks(p.pairs);
    const size_t lds = (size_t)kRouteWaves * ((experts + 1) & ~1) * sizeof(uint16_t);
    p.chunk = (p.pairs + blocks - 1) / blocks;
    p.chunk = (p.chunk + kRouteThreads - 1) / kRouteThreads * kRouteThreads;
    p.blocks = (int)blocks;
    const u32 groups = tokens_q ? tokens_q->total_groups : 0;
    const unsigned all = (unsigned)blocks + groups / kRouteQuantGroups + (groups % kRouteQuantGroups != 0);
    const GroupRows q = tokens_q ? *tokens_q : GroupRows{};
    if (blocks == 1) {
        hipLaunchKernelGGL(route_place_kernel<true>, dim3(all), dim3(kRouteThreads), lds, st, p, q);
    } else {
        // (the quantiser's workgroups all behind the placing: some of them beside the counting, whose end the placing waits for, took 0.4 to 3 us more a call
        // at 200 to 4096 tokens of 128 x 2048 x 768, 32 x 3584 x 1536 and 64 x 1024 x 512, the same at 8192)
        hipLaunchKernelGGL(route_count_kernel, dim3((unsigned)blocks), dim3(kRouteThreads), 0, st, p);
        hipLaunchKernelGGL(route_place_kernel<false>, dim3(all), dim3(kRouteThreads), lds, st, p, q);
    }
    return check_launch("route_tokens");
}

}  // namespace cfp8

extern "C" int cfp8_route_tokens(const void* indices, int index_bytes, const uint8_t* token_mask, int64_t tokens, int topk, int experts,
                                 int64_t alignment, int flags, int64_t capacity, int32_t* row_tokens, int32_t* row_experts,
                                 int32_t* row_map, int64_t* slot_order, const void* weights, int weights_dtype, void* sorted_weights,
                                 int32_t* m_sizes, int32_t* m_offsets, void* workspace, size_t workspace_bytes, void* stream) {
    return cfp8::route_and_quantise(indices, index_bytes, token_mask, tokens, topk, experts, alignment, flags, capacity, row_tokens, row_experts, row_map, slot_order,
                                    weights, weights_dtype, sorted_weights, m_sizes, m_offsets, workspace, workspace_bytes, nullptr, static_cast<hipStream_t>(stream));
}
