// Interface of the ring GEMM (gemm_ring.hip) to the entry points.
#pragma once

#include "cfp8_common.h"

namespace cfp8 {

// kRingGateUp, kRingDown: block-scaled products of MoE experts on rows that lie expert behind expert; the first one gathers its
// rows from the tokens and ends in SwiGLU
enum : int { kRingRow = 0, kRingBlock = 1, kRingMx = 2, kRingGateUp = 3, kRingDown = 4 };
constexpr int kRingGroupRows = 64;

struct RingArgs {
    const uint8_t* a;      // activations e4m3 [M, K]
    const uint8_t* w;      // weights e4m3 [N, K], kRingMx: packed e2m1 [N, K / 2]
    const uint8_t* ws;     // kRingMx: e8m0 [N, K / 32]
    const float* sa;       // [M]; kRingBlock: [M, K / 128]
    const float* sb;       // kRingRow: [N]; kRingBlock: see the strides
    const uint16_t* bias;  // bf16 [N] or null
    void* out;
    float* partial;        // [slices, M, N] when slices > 1
    int64_t ld_a, ld_w, ld_ws, ld_out, sb_stride_n, sb_stride_k;
    const int32_t* row_tokens;  // kRingGateUp: the token of every row; M is then the number of tokens
    const int32_t* sizes;       // kRingGateUp, kRingDown: rows of every expert, and their inclusive cumulative sum
    const int32_t* ends;
    int experts;
    int M, N, K;
    int tiles_m, tiles_n, slices, slice_steps;
};

struct RingPlan {
    int bm, bn, slices;
    double cost;           // microseconds, estimated
};
RingPlan ring_plan(int mode, int64_t M, int64_t N, int64_t K, size_t partial_bytes, int cus);
bool ring_takes(int mode, const RingArgs& p, int out_dtype);  // whether the operands fit what the kernel assumes
// the form for few rows, all of K a workgroup, in place of `plan` and of every other file's kernel: strips of 16 weight rows a workgroup, 0: not
int ring_few_first(int mode, const RingArgs& p, const RingPlan& plan);
int launch_ring_few(int mode, RingArgs& p, int strips, int out_dtype, hipStream_t st);
// the linear of up to four tokens (K <= 4096, one token 8192, a multiple of 128) as one launch of streams: waves a workgroup, 0: other kernels are ahead
int linear_stream_waves(int mode, int64_t M, int64_t N, int64_t K);
int launch_linear_stream(int mode, const RingArgs& p, const void* x, int64_t ld_x, int waves, int out_dtype, hipStream_t st);
bool ring_grouped_takes(int64_t K);
int launch_ring_grouped(int mode, RingArgs& p, int64_t row_tiles, bool once, hipStream_t st);
int launch_ring(int mode, RingArgs& p, const RingPlan& plan, int out_dtype, hipStream_t st);

}  // namespace cfp8
