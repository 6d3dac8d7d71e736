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
// What bounds it: nothing but latency - 65536 pairs are half a megabyte of indices and outputs of the same size.  The
// same layout built from library calls (a stable argsort, a scatter-add for the counts, a sort along the slots,
// gathers, comparisons and fills, each over 10^2 .. 10^5 elements) is some thirty launches of 2 .. 45 us each:
// 230-250 us at every size from 16 to 8192 tokens, top 8 of 128 experts, against 7.6 us (16 tokens) and 4.8 + 11.9 us (8192 tokens) here.
#include "cfp8_common.h"

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
};

// expert of a pair; `experts` for a pair that goes nowhere (masked token, index out of range)
__device__ __forceinline__ bool route_masked(const RouteArgs& p, int64_t token) { return p.mask && !p.mask[token]; }
__device__ __forceinline__ int route_expert(const RouteArgs& p, bool masked, int64_t pair) {
    if (masked) return p.experts;
    const int64_t e = p.idx64 ? static_cast<const int64_t*>(p.indices)[pair] : (int64_t) static_cast<const int32_t*>(p.indices)[pair];
    return e >= 0 && e < p.experts ? (int)e : p.experts;
}

__device__ __forceinline__ void route_histogram(const RouteArgs& p, int* hist, int64_t first, int64_t last) {
    const int t = threadIdx.x;
    for (int e = t; e < p.experts; e += kRouteThreads) hist[e] = 0;
    __syncthreads();
    for (int64_t i = first + t; i < last; i += kRouteThreads) {
        const int e = route_expert(p, route_masked(p, i / p.topk), i);
        if (e < p.experts) atomicAdd(&hist[e], 1);
    }
    __syncthreads();
}

__global__ __launch_bounds__(kRouteThreads) void route_count_kernel(const RouteArgs p) {
    __shared__ int hist[kRouteMaxExperts];
    const int64_t first = (int64_t)blockIdx.x * p.chunk;
    route_histogram(p, hist, first, first + p.chunk < p.pairs ? first + p.chunk : p.pairs);
    for (int e = threadIdx.x; e < p.experts; e += kRouteThreads) p.hist[(int64_t)blockIdx.x * p.experts + e] = hist[e];
}

template <bool ONE>
__global__ __launch_bounds__(kRouteThreads) void route_place_kernel(const RouteArgs p) {
    __shared__ int total[kRouteMaxExperts];   // pairs of every expert
    __shared__ int base[kRouteMaxExperts];    // next row of every expert for this workgroup
    __shared__ int ends[kRouteMaxExperts];    // inclusive cumulative group ends
    __shared__ int wave_sum[kRouteWaves];
    extern __shared__ uint16_t counts[];      // [wave][experts rounded up to even]
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int E = p.experts, EP = (E + 1) & ~1;
    const int64_t first = (int64_t)blockIdx.x * p.chunk;
    const int64_t last = first + p.chunk < p.pairs ? first + p.chunk : p.pairs;
    if (ONE) {
        route_histogram(p, total, 0, p.pairs);
        for (int e = t; e < E; e += kRouteThreads) base[e] = 0;
        __syncthreads();
    } else {
        for (int e = t; e < E; e += kRouteThreads) total[e] = 0, base[e] = 0;
        __syncthreads();
        // thread (part, expert): the workgroups' histograms are read in parallel, kRouteThreads words at a time
        const int n = (int)gridDim.x * E;
        for (int i = t; i < n; i += kRouteThreads) {
            const int c = p.hist[i];
            if (c) {
                const int b = i / E, e = i - b * E;
                atomicAdd(&total[e], c);
                if (b < (int)blockIdx.x) atomicAdd(&base[e], c);
            }
        }
        __syncthreads();
    }
    // padded group sizes and their inclusive prefix sum, one expert per thread
    {
        int64_t size = 0;
        if (t < E) {
            size = total[t];
            if ((p.flags & CFP8_ROUTE_KEEP_EMPTY) && size < p.alignment) size = p.alignment;
            size = (size + p.alignment - 1) / p.alignment * p.alignment;
        }
        int run = (int)size;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int v = __shfl_up(run, off);
            if (lane >= off) run += v;
        }
        if (lane == 63) wave_sum[wave] = run;
        __syncthreads();
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
        const int64_t pair = i0 + t;
        const bool have = pair < last;
        const int64_t token = have ? pair / p.topk : 0;
        const bool masked = have && route_masked(p, token);
        const int e = have ? route_expert(p, masked, pair) : E;
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
            p.row_tokens[row] = (int32_t)token;
            if (p.row_experts) p.row_experts[row] = e;
        }
        if (have) {
            // the pair's place among its token's slots, ascending by expert, slots of one expert in their order
            const int64_t slot0 = token * p.topk;
            const int s = (int)(pair - slot0);
            int place = 0;
            for (int k = 0; k < p.topk; ++k) {
                const int o = route_expert(p, masked, slot0 + k);
                place += o < e || (o == e && k < s);
            }
            p.row_map[slot0 + place] = row;
            if (p.slot_order) p.slot_order[slot0 + place] = s;
            if (p.sorted_weights)
                p.sorted_weights[slot0 + place] = p.w32 ? (uint16_t)(pack_bf16x2(static_cast<const float*>(p.weights)[pair], 0.f) & 0xFFFFu)
                                                        : static_cast<const uint16_t*>(p.weights)[pair];
        }
        __syncthreads();
        if (t < E) base[t] += added;
        // (the next round's first barrier orders this against its readers)
    }
    // padding: the rows behind every group's last pair, and the rows past the last group
    // (a wave per expert: the whole workgroup on one expert after the other took 25 us for 128 of them)
    for (int e = blockIdx.x * kRouteWaves + wave; e < E; e += gridDim.x * kRouteWaves) {
        const int end = ends[e], start = e ? ends[e - 1] : 0;
        for (int64_t r = start + (int64_t)total[e] + lane; r < end && r < p.capacity; r += 64) {
            p.row_tokens[r] = -1;
            if (p.row_experts) p.row_experts[r] = e;
        }
    }
    for (int64_t r = (int64_t)ends[E - 1] + (int64_t)blockIdx.x * kRouteThreads + t; r < p.capacity; r += (int64_t)gridDim.x * kRouteThreads) {
        p.row_tokens[r] = (p.flags & CFP8_ROUTE_END_NOT_PADDING) ? 0x7FFFFFFF : -1;
        if (p.row_experts) p.row_experts[r] = -1;
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

extern "C" int cfp8_route_tokens(const void* indices, int index_bytes, const uint8_t* token_mask, int64_t tokens, int topk, int experts,
                                 int64_t alignment, int flags, int64_t capacity, int32_t* row_tokens, int32_t* row_experts,
                                 int32_t* row_map, int64_t* slot_order, const void* weights, int weights_dtype, void* sorted_weights,
                                 int32_t* m_sizes, int32_t* m_offsets, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace cfp8;
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
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t blocks = route_blocks(p.pairs);
    const size_t lds = (size_t)kRouteWaves * ((experts + 1) & ~1) * sizeof(uint16_t);
    p.chunk = (p.pairs + blocks - 1) / blocks;
    p.chunk = (p.chunk + kRouteThreads - 1) / kRouteThreads * kRouteThreads;
    if (blocks == 1) {
        hipLaunchKernelGGL(route_place_kernel<true>, dim3(1), dim3(kRouteThreads), lds, st, p);
    } else {
        hipLaunchKernelGGL(route_count_kernel, dim3((unsigned)blocks), dim3(kRouteThreads), 0, st, p);
        hipLaunchKernelGGL(route_place_kernel<false>, dim3((unsigned)blocks), dim3(kRouteThreads), lds, st, p);
    }
    return check_launch("route_tokens");
}
