// What the GEMM translation units of libcosmosfp8 share: the argument block of every GEMM kernel, the launch
// record behind cfp8_gemm_dispatch_info, and a few device helpers.
#pragma once

#include <atomic>

#include "cfp8_common.h"

namespace cfp8 {

enum : int { kRowwise = 0, kBlock = 1, kGrouped = 2 };

struct GemmArgs {
    const uint8_t* a;   // activations fp8 [M, K]
    const uint8_t* b;   // weights fp8 [N, K] (grouped: [E, N, K])
    const float* sa;    // rowwise [M]; block [M, K/128]
    const float* sb;    // rowwise [N]; block: see strides
    const int32_t* m_indices;
    void* out;
    int64_t ld_a, ld_b, ld_out;
    int64_t sb_stride_n, sb_stride_k, sb_stride_e;
    int M, N, K;
    int tiles_m, tiles_n;
    // split-K (rowwise, at most 64 tokens): fp32 partial sums [k_slices, M, N] in caller-provided memory
    float* partial;
    size_t partial_bytes;
    int k_slices, slice_steps;
    // grouped GEMM with the SwiGLU + 1x128 quantisation epilogue: scales of the quantised product [M, N / 256]
    float* h_scales;
    int64_t ld_hs;
    // gemm_grouped_xres_kernel: pieces along N of the tile rows that are not whole-row units
    int unit_parts;
    // gemm_rowwise_256p_kernel: tiles of the last, at most half-full round, computed as quarter tiles by all workgroups
    int tail_tiles;
    // gemm_rowwise_edge_kernel: bf16 [N] or null; quarter tiles below the last row of tiles and beside their last column
    const uint16_t* bias;
    int edge_rows, edge_cols;
};

// ---- host side (gemm_fp8.hip) ---------------------------------------------
bool dry_run();                                                                   // launches are being recorded, not made
bool note_launch(const char* kernel, unsigned grid, unsigned block, size_t lds);  // true: launch for real
int raise_lds_limit(const void* fn, size_t lds, std::atomic<bool>& flag);         // once per (device, function)
int device_slot();                                                                // 0..63, 64 = not cached
int cu_count();                                                                   // compute units of the current device
// what cfp8_gemm_mxfp4 (`split`: cfp8_gemm_mxfp4_split; `linear`: cfp8_linear_mxfp4) launches for a problem, with every operand at `any`; while dry_run()
int mx4_dispatch(const void* any, int64_t M, int64_t N, int64_t K, int out_dtype, bool split, size_t partial_bytes, bool linear);
size_t block_partial_bytes(int64_t M, int64_t N, int64_t K);                      // of the block-scaled product's slices of K

// ---- gemm_experts.hip
struct ExpertsArgs {
    const uint8_t* x;            // fp8: gate_up the tokens [tokens, K], down the rows [rows, K]
    const float* xs;             // [tokens or rows, K / 128]
    const uint8_t* w;            // [experts, N, K], gate_up: gate and up rows in turn, 16 at a time
    const float* ws;             // [experts, N / 128, K / 128]
    const int32_t* row_tokens;   // [rows], negative: a row of padding
    const int32_t* row_experts;  // [rows]
    const int32_t* rows_end;     // rows that the groups take
    uint8_t* h;                  // gate_up: [rows, N / 2] fp8
    float* hs;                   // gate_up: [rows, N / 256]
    uint16_t* out;               // down: [rows, N] bf16
    int tokens, N, K, tiles_m, tiles_n;
    int whole_tiles;             // gate_up: halves of tiles that are padding are written, for a down product of another kernel, which reads them
};
bool experts_gate_up_takes(int64_t tokens, int64_t hidden, int64_t inter);
bool experts_down_takes(int64_t hidden, int64_t inter);
int launch_experts_gate_up(ExpertsArgs& p, int64_t rows, bool once, hipStream_t st);
int launch_experts_down(ExpertsArgs& p, int64_t rows, bool once, hipStream_t st);

// ---- units of the kernels in which a workgroup walks rows of tiles ----------
// The schedule for tiles_m tile rows of tiles_n tiles on `cus` workgroups: one workgroup per CU.  Tile rows beyond the
// last full round of whole rows (all of them, with fewer tile rows than CUs) are cut along N into `parts` pieces; a
// unit costs its tiles plus `unit_cost` tiles for starting it, and `parts` is the count with the shortest last round.  `fill` is the share of the run's tile slots (CUs x length of the longest workgroup's run) that hold tiles.
struct UnitPlan {
    int parts;
    int64_t blocks;
    double fill;
};
inline UnitPlan unit_plan(int tiles_m, int tiles_n, int cus, int unit_cost) {
    const int rem = tiles_m >= cus ? tiles_m % cus : tiles_m;
    int parts = 1;
    int64_t span = (int64_t)(tiles_m / cus) * (tiles_n + unit_cost);
    if (rem) {
        int64_t best = INT64_MAX;
        for (int q = 1; q <= tiles_n; ++q) {
            const int64_t rounds = ((int64_t)rem * q + cus - 1) / cus;
            const int64_t cost = rounds * ((tiles_n + q - 1) / q + unit_cost);
            if (cost < best) best = cost, parts = q;
        }
        span += best;
    }
    const int64_t units = (int64_t)(tiles_m - rem) + (int64_t)rem * parts;
    int64_t blocks = units < cus ? units : cus;
    // (the kernel takes tiles_m / gridDim.x * gridDim.x tile rows for whole-row units: with fewer tile rows than CUs
    // the grid must exceed the tile rows unless every unit is a whole row anyway)
    if (tiles_m < cus && parts == 1) blocks = tiles_m;
    return {parts, blocks, (double)tiles_m * tiles_n / ((double)cus * (double)span)};
}

// gemm_grouped_xres.hip
int launch_grouped_xres(GemmArgs& p, int out_dtype, hipStream_t st);
bool grouped_xres_pays(const GemmArgs& p);  // enough of the CUs' tile slots would hold tiles

// ---- device side ------------------------------------------------------------
#define CFP8_PHASE_END() __builtin_amdgcn_sched_barrier(0)
// Wait until at most `vm` of this wave's loads are outstanding and its LDS reads are done, then the workgroup barrier.
// Written out as instructions: in front of a barrier it knows of, the compiler waits for every load it has issued,
// including the direct-to-LDS loads that are meant to stay in flight across the barrier.
#define CFP8_WAIT_BARRIER(vm) asm volatile("s_waitcnt vmcnt(" #vm ") lgkmcnt(0)\n\ts_barrier" ::: "memory")

// A 16-byte buffer store with a scalar offset.  The store reads its data registers a while after it has been issued, and a VALU
// instruction right behind it that writes one of them reaches memory in its place for some of the lanes (seen on gfx950
// where L2 was full of lines to write back: lanes 12 .. 15 of every 16 stored the result of the next instruction).  One
// instruction in between is enough; the compiler keeps that distance for stores without a scalar offset only.
__device__ __forceinline__ void buffer_store16(u32x4 v, __amdgpu_buffer_rsrc_t r, uint32_t lane_offset, uint32_t offset) {
    __builtin_amdgcn_raw_buffer_store_b128(v, r, lane_offset, offset, 0);
    asm volatile("s_nop 1" ::"v"(v));
}

// One int of a table that the kernel does not write, by a scalar load.  Behind the first store of a kernel the compiler turns
// such a read into a vector load, and then waits for every load in flight, the direct-to-LDS ones included.
__device__ __forceinline__ int scalar_table_load(const int32_t* table, int index) {
    const int32_t* const ptr = table + index;  // uniform
    int v;
    asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(ptr) : "memory");
    return v;
}

// Workgroup id -> (tile_m, tile_n).  Consecutive workgroup ids are dealt round
// robin to the 8 XCDs, each with its own L2: give every XCD one contiguous range
// of tiles, and walk a range in bands of GM tile-rows so that co-resident
// workgroups share activation rows and weight rows in that L2.
// GM: tile-rows per band.  8 for the dense problems; the grouped kernels take kGroupedBandRows = 4, about the
// tile-rows of one expert at the MoE shapes served here (an expert's weight tile is then shared by the
// workgroups of one band: FETCH_SIZE of the K = 768 down projection of 128 experts falls from 1.34 to 1.10
// times its operand bytes, run time unchanged).
constexpr int kGroupedBandRows = 4;
template <int GM = 8>
__device__ __forceinline__ void tile_of_block(int pid, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int total = tiles_m * tiles_n;
    const int xcd = pid & 7, local = pid >> 3;
    const int base = total >> 3, rem = total & 7;
    const int lin = xcd * base + (xcd < rem ? xcd : rem) + local;
    const int band = GM * tiles_n;
    const int g = lin / band, first = g * GM;
    const int gsz = (tiles_m - first) < GM ? (tiles_m - first) : GM;
    const int in = lin - g * band;
    tm = first + in % gsz;
    tn = in / gsz;
}

}  // namespace cfp8
