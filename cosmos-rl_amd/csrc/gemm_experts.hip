// The two products of a MoE layer's experts with many rows:
//
//   gate_up  from the quantised tokens to the quantised hidden activation: h[r, c] = bf16(bf16(silu(gate)) * up) of row r's token
//            and expert, requantised 1x128
//   down     from that to bf16 rows
//
// Rows lie expert by expert, every group padded to 128 of them (row_tokens < 0: padding, whose operands arrive as zeros); the
// weight's gate and up rows alternate in units of 16 (one MFMA tile), so that a 128 x 256 tile holds both halves of one 1x128 group
// of h.  One workgroup of eight waves a CU (2 x 4, wave tiles of 64 x 64) walks tiles b, b + gridDim.x, ...; the K steps of
// consecutive tiles form one stream of loads, so that a tile begins on operands that arrived under the one before.
//
// K step kt, four token tiles (x) and four weight tiles (w) a wave, all of whose sixteen raw products have registers of their own:
//
//   A  MFMAs of x tiles 0 and 1; the products of x tiles 2 and 3 of the step before are scaled and added; reads of x fragments 2, 3
//   barrier: tile kt + 1 has landed in every wave's view, every wave has read tile kt
//   B  MFMAs of x tiles 2 and 3; the products of x tiles 0 and 1 are added; the next step's fragments and scales, each weight
//      fragment behind its last MFMA; loads of tile kt + 3 into the stage that tile kt has left
//
// Both operands go from global memory straight into LDS, rows of the tokens wherever they lie, through a ring of three stages.
// The activation scales come the same way, eight K steps of 128 rows at a time.  Products are scaled and added in the order of K
// as in the other block-scaled kernels, and have their bits.
//
// What bounds it (8192 tokens, top 8 of 128 experts of 2048 x 768; gemm_block_w8p_kernel in its place takes 295 us and 635
// thousand cycles, this one 259 us and 525 thousand): instructions.  That kernel's time hardly moved when its loads, its SwiGLU or three
// quarters of its FMAs were taken out one at a time, or when the SwiGLU ran under the next tile's K steps: a step has 16 MFMAs a wave
// in some 270 instructions, and every wave waits at the same barrier for the slowest to issue them.  Here a step has 185 (no
// choices by scalar selects: the last three steps, which load the next tile, are code of their own; no detour of the scales
// through registers), and MFMAs follow the barrier at once, since no product waits for an addition to free its registers.
// Gathering the rows saves the padded copy of the tokens: 28 us of 38 for a quantiser that writes each token eight times.
// The down product (165 us, 268 MB written) is bound by its stores among the loads: 119 us without the stores, 113 without the loads, 105
// without either; neither their cache policy, nor tiles that are contiguous in memory, nor stores behind the next loads change that.
//
// A wave whose 64 rows are all padding only loads and keeps the barriers (48 rows an expert: 178 -> 167 us a call), and those rows of
// h are neither written nor read (152.4 -> 147.1 us), unless the down product is another kernel's (ExpertsArgs::whole_tiles).
#include <atomic>
#include <type_traits>

#include "gemm_internal.h"

namespace cfp8 {

constexpr int kExBM = 128, kExBN = 256, kExStages = 3;
constexpr int kExXS = kExBM * 128, kExStage = kExXS + kExBN * 128;
constexpr int kExScales = kExStages * kExStage;            // activation scales: three buffers of [128 rows][8 steps]
constexpr int kExExchange = kExScales + 3 * kExBM * 32;    // the four waves' maxima of every row
constexpr int kExWeightScales = kExExchange + kExBM * 16;  // [two tiles][K step][gate, up]
constexpr int kExTokens = kExWeightScales + 2 * 64 * 4;    // the next tile's row_tokens
constexpr int kExLds = kExTokens + kExBM * 4;
constexpr uint32_t kExOutside = 0xF0000000u;  // a per-lane offset past the end of every buffer: loads give zeros, stores are dropped

// four registers (one a row tile) of four lanes l, l + 16, l + 32, l + 48: lane quarter q's register j becomes lane quarter j's register q
__device__ __forceinline__ void quarters_transpose(u32 (&v)[4]) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const u32x2 a = __builtin_amdgcn_permlane32_swap(v[k], v[k + 2], false, false);
        v[k] = a[0];
        v[k + 2] = a[1];
    }
#pragma unroll
    for (int k = 0; k < 4; k += 2) {
        const u32x2 a = __builtin_amdgcn_permlane16_swap(v[k], v[k + 1], false, false);
        v[k] = a[0];
        v[k + 1] = a[1];
    }
}

// ONCE: the weights are loaded as a stream
template <bool DOWN, bool ONCE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void gemm_experts_kernel(const ExpertsArgs p) {
    constexpr int XS = kExXS, STAGE = kExStage;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    typedef __attribute__((address_space(3))) void lds_void;
    // (tiles are dealt to the XCDs in contiguous ranges: those of padding behind the last group, up to the bound, would all be the last XCD's)
    const int bound = p.tiles_m, held = scalar_table_load(p.rows_end, 0) >> 7;
    const int tiles_m = held < bound ? held : bound;
    const int ntiles = tiles_m * p.tiles_n;
    int pid = blockIdx.x;
    if (pid >= ntiles) return;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave >> 2, wn = wave & 3;  // (a SIMD has a wave of either half of the rows)
    const int lrow = lane & 15, quarter = lane >> 4;
    const int KT = p.K >> 7;
    __builtin_assume(KT >= 4 && KT <= 32);
    const int G = (KT + 7) >> 3;  // groups of eight K steps

    // ---- loads.  Load i of a wave: rows (wave + 8 i) * 8 .. + 7 of the tile, 16-byte chunk c of row r at position c ^ f(r).
    const uint32_t chunk = (uint32_t)(((lane & 7) ^ ((wave & 1) * 4 + ((lane >> 4) & 1))) << 4);
    // gate_up: all tokens, whose rows the lanes pick; down: the tile's first 64 or 128 rows
    auto x_rsrc = [&](int m0, int rows) {
        return DOWN ? __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.x) + (int64_t)m0 * p.K, 0, rows * p.K, 0x00020000)
                    : __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.x), 0, (int)((uint32_t)p.tokens * (uint32_t)p.K), 0x00020000);
    };
    auto xs_rsrc = [&](int m0, int rows) {
        return DOWN ? __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.xs) + (int64_t)m0 * KT, 0, rows * KT * 4, 0x00020000)
                    : __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.xs), 0, (int)((uint32_t)p.tokens * (uint32_t)KT * 4u), 0x00020000);
    };
    uint32_t vw[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) vw[i] = (uint32_t)((wave + 8 * i) * 8 + (lane >> 3)) * (uint32_t)p.K + chunk;
    uint32_t vx[2], vxs[2];  // of the tile that is being loaded
    auto set_rows = [&](int i, int token) {
        vx[i] = token >= 0 ? (uint32_t)token * (uint32_t)p.K + chunk : kExOutside;
        vxs[i] = token >= 0 ? (uint32_t)(token * KT + (lane & 7)) * 4u : kExOutside;
    };
    // `rows`: 64 where the second half of the tile is padding, whose rows down does not read (a group's padding follows its rows)
    auto place = [&](int id, int& m0, int& n0, __amdgpu_buffer_rsrc_t& rw, int& expert, int& rows) {
        int tm, tn;
        tile_of_block<kGroupedBandRows>(id, tiles_m, p.tiles_n, tm, tn);
        m0 = tm * kExBM;
        n0 = tn * kExBN;
        const int32_t *const at = p.row_experts + m0, *const half = p.row_tokens + m0 + 64;  // (a group's rows begin on a multiple of 128)
        int token;
        asm volatile("s_load_dword %0, %2, 0x0\n\ts_load_dword %1, %3, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=&s"(expert), "=&s"(token) : "s"(at), "s"(half) : "memory");
        rows = token < 0 ? 64 : kExBM;
        // (down: weight rows beyond N, where N is an odd multiple of 128, arrive as zeros)
        rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w) + ((int64_t)expert * p.N + n0) * p.K, 0,
                                               (p.N - n0 < kExBN ? p.N - n0 : kExBN) * p.K, 0x00020000);
    };
    auto dma_x = [&](__amdgpu_buffer_rsrc_t r, int kt, int stage, int i) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)(smem + stage + (wave + 8 * i) * 1024), 16, vx[i], (uint32_t)kt << 7, 0, 0);
    };
    auto dma_w = [&](__amdgpu_buffer_rsrc_t r, int kt, int stage, int i) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)(smem + stage + XS + (wave + 8 * i) * 1024), 16, vw[i], (uint32_t)kt << 7, 0, ONCE ? 2 : 0);
    };
    auto dma_scales = [&](__amdgpu_buffer_rsrc_t r, int group, int buf) {  // (steps beyond K: the next token's, never used)
#pragma unroll
        for (int i = 0; i < 2; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)(smem + kExScales + buf * (kExBM * 32) + (wave + 8 * i) * 256), 4, vxs[i], (uint32_t)group * 32u, 0, 0);
    };
    auto dma_weight_scales = [&](int expert, int n0, int par) {  // one wave
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.ws) + ((int64_t)expert * (p.N >> 7) + (n0 >> 7)) * KT, 0,
                                                                           (p.N - n0 < kExBN ? 1 : 2) * KT * 4, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)(smem + kExWeightScales + par * 256), 4, (uint32_t)((lane & 1) * KT + (lane >> 1)) * 4u, 0, 0, 0);
    };

    // ---- reads
    const int fsw = ((lrow >> 1) & 1) | (((lrow >> 3) & 1) << 2);
    const int c1 = ((2 * quarter) ^ fsw) << 4;
    const int x_at = (wm * 64 + lrow) * 128 + c1, w_at = XS + (wn * 64 + lrow) * 128 + c1;
    auto frag = [&](int at, int tile16) {  // (the lane's second chunk is the other one of an even and odd pair)
        const i32x4 lo = *reinterpret_cast<const i32x4*>(smem + at + tile16 * 2048);
        const i32x4 hi = *reinterpret_cast<const i32x4*>(smem + (at ^ 16) + tile16 * 2048);
        return i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    i32x8 W[4], X[4];
    float sm[4];
    u32x2 sn;  // gate_up: weight scales of the gate and of the up rows; down: the first is that of the wave's rows
    const int s_at = kExScales + (wm * 64 + lrow) * 32;
    auto read_scales = [&](int buf, int par, int kt) {
        const float* const at = reinterpret_cast<const float*>(smem + s_at + buf * (kExBM * 32) + (kt & 7) * 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) sm[j] = at[j * 16 * 8];
        if (DOWN) sn[0] = *reinterpret_cast<const u32*>(smem + kExWeightScales + par * 256 + kt * 8 + (wn >> 1) * 4);
        else sn = *reinterpret_cast<const u32x2*>(smem + kExWeightScales + par * 256 + kt * 8);
    };

    int m0, n0, expert, rows;
    __amdgpu_buffer_rsrc_t rw;
    place(pid, m0, n0, rw, expert, rows);
    __amdgpu_buffer_rsrc_t rx = x_rsrc(m0, rows), rxs = xs_rsrc(m0, rows);
    bool idle = wm == 1 && rows < kExBM;  // this wave has no rows
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = (wave + 8 * i) * 8 + (lane >> 3);
        set_rows(i, DOWN ? row : p.row_tokens[m0 + row]);
    }
    if (wave == 0) dma_weight_scales(expert, n0, 0);
    dma_scales(rxs, 0, 0);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
#pragma unroll
        for (int i = 0; i < 2; ++i) dma_x(rx, k, k * STAGE, i);
#pragma unroll
        for (int i = 0; i < 4; ++i) dma_w(rw, k, k * STAGE, i);
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");

    f32x4 acc[4][4], P[4][4];  // [w tile][x tile]
    float sc2[2], sc3[2];      // scales of x tiles 2 and 3 (gate, up) that go with the products waiting in P
    int stage = 0;             // of the stream's current step, in bytes
    int gb = 0, par = 0;       // the tile's first buffer of activation scales, its weight scales
// (the empty statement pins the FMAs to this place)
#define CFP8_PRODUCT(i, j) P[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(W[i], X[j], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0)
    auto add = [&](int i, int j, float sc, bool first) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j][e] = __builtin_fmaf(P[i][j][e], sc, first ? 0.f : acc[i][j][e]);
        asm volatile("" : "+v"(acc[i][j]));
    };
    // three buffers of activation scales, one a group
    auto buffer_of = [&](int g) {
        const int b = gb + g;
        return b >= 6 ? b - 6 : b >= 3 ? b - 3 : b;
    };
    for (;;) {
        const int pid_n = pid + (int)gridDim.x;
        const bool has_next = pid_n < ntiles;
        int m0n, n0n, expert_n, rows_n;
        __amdgpu_buffer_rsrc_t rwn;
        place(has_next ? pid_n : pid, m0n, n0n, rwn, expert_n, rows_n);  // (no next tile: this one's first steps are fetched once more)
        const __amdgpu_buffer_rsrc_t rxn = x_rsrc(m0n, rows_n), rxsn = xs_rsrc(m0n, rows_n);

        // what a step loads beside its tile, in front of it: the next barrier waits for it
        auto beside = [&](int kt, auto first_c, auto left_c) {
            constexpr bool first = decltype(first_c)::value;
            constexpr int left = decltype(left_c)::value;
            if constexpr (first && !DOWN) {
                if (wave < 2) {
                    const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(p.row_tokens) + m0n + wave * 64, 0, 256, 0x00020000);
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rt, (lds_void*)(smem + kExTokens + wave * 256), 4, (uint32_t)lane * 4u, 0, 0, 0);
                }
            } else if constexpr (left == 3) {
                if ((kt & 7) == 4 && kt < 8 * (G - 1)) dma_scales(rxs, (kt >> 3) + 1, buffer_of((kt >> 3) + 1));
            } else if constexpr (left == 2) {
                if constexpr (!DOWN) {
                    const int32_t* const tok = reinterpret_cast<const int32_t*>(smem + kExTokens) + wave * 8 + (lane >> 3);
                    set_rows(0, tok[0]);
                    set_rows(1, tok[64]);
                }
                dma_scales(rxsn, 0, buffer_of(G));
                if (wave == 0) dma_weight_scales(expert_n, n0n, par ^ 1);
            }
        };
        // tile kt + 1 has landed when at most the six loads of the step before are outstanding, and the stores of the tile before:
        // gate_up three behind the loads of its last step, down eight in front of those of this tile's third
        auto wait = [&](auto first_c) {
            if constexpr (decltype(first_c)::value && DOWN) CFP8_WAIT_BARRIER(14);
            else if constexpr (decltype(first_c)::value) CFP8_WAIT_BARRIER(9);
            else CFP8_WAIT_BARRIER(6);
        };
        // a step of a wave without rows: it loads as the others do
        auto step_idle = [&](int kt, auto first_c, auto left_c) {
            constexpr int left = decltype(left_c)::value;
            const int kl = left == 3 ? kt + 3 : 2 - left;
            wait(first_c);
            CFP8_PHASE_END();
            beside(kt, first_c, left_c);
            CFP8_PHASE_END();
            if constexpr (!DOWN || left > 0) {
                dma_x(left == 3 ? rx : rxn, kl, stage, 0);
                dma_x(left == 3 ? rx : rxn, kl, stage, 1);
#pragma unroll
                for (int i = 0; i < 4; ++i) dma_w(left == 3 ? rw : rwn, kl, stage, i);
            }
            CFP8_PHASE_END();
            stage = stage == 2 * STAGE ? 0 : stage + STAGE;
        };
        // LEFT: K steps behind this one, 3 for all but the last three
        auto step = [&](int kt, auto first_c, auto left_c) {
            constexpr bool first = decltype(first_c)::value;
            constexpr int left = decltype(left_c)::value;
            const int next = stage == 2 * STAGE ? 0 : stage + STAGE;
            const int xc = x_at + stage, xn = x_at + next, wn_ = w_at + next;
            const int kl = left == 3 ? kt + 3 : 2 - left;  // the step to load, of the next tile in the last three
            const __amdgpu_buffer_rsrc_t r = left == 3 ? rw : rwn, ra = left == 3 ? rx : rxn;
            constexpr bool loads = !DOWN || left > 0;  // (down: the last step's follow the epilogue, which takes the stage)
            X[2] = frag(xc, 2);
            CFP8_PHASE_END();
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                CFP8_PRODUCT(i, 0);
                if (!first) add(i, 2, sc2[i & 1], false);
                if (i == 0) X[3] = frag(xc, 3);
                CFP8_PHASE_END();
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                CFP8_PRODUCT(i, 1);
                if (!first) add(i, 3, sc3[i & 1], false);
                CFP8_PHASE_END();
            }
            wait(first_c);
            CFP8_PHASE_END();
            CFP8_PRODUCT(0, 2);
            CFP8_PRODUCT(0, 3);
            CFP8_PHASE_END();
            float sc0[2], sc1[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const float s = __uint_as_float(sn[DOWN ? 0 : u]);
                sc0[u] = sm[0] * s;
                sc1[u] = sm[1] * s;
                sc2[u] = sm[2] * s;
                sc3[u] = sm[3] * s;
            }
            beside(kt, first_c, left_c);
            CFP8_PHASE_END();
            if (left > 0) {
                W[0] = frag(wn_, 0);
                X[0] = frag(xn, 0);
            }
            if (loads) dma_x(ra, kl, stage, 0);
            CFP8_PHASE_END();
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i < 3) CFP8_PRODUCT(i + 1, 2);
                add(i, 0, sc0[i & 1], first);
                if (i < 3) CFP8_PRODUCT(i + 1, 3);
                add(i, 1, sc1[i & 1], first);
                CFP8_PHASE_END();
                if (i < 3 && left > 0) W[i + 1] = frag(wn_, i + 1);
                if (i == 0) {
                    if (left > 0) X[1] = frag(xn, 1);
                    if (loads) dma_x(ra, kl, stage, 1);
                }
                if (i == 1 && left > 0) read_scales(buffer_of((kt + 1) >> 3), par, kt + 1);
                if (loads) dma_w(r, kl, stage, i);
                CFP8_PHASE_END();
            }
            stage = next;
        };
        using yes = std::integral_constant<bool, true>;
        using no = std::integral_constant<bool, false>;
        auto tile = [&](auto& one) {
            one(0, yes{}, std::integral_constant<int, 3>{});
            for (int kt = 1; kt < KT - 3; ++kt) one(kt, no{}, std::integral_constant<int, 3>{});
            one(KT - 3, no{}, std::integral_constant<int, 2>{});
            one(KT - 2, no{}, std::integral_constant<int, 1>{});
            one(KT - 1, no{}, std::integral_constant<int, 0>{});
        };
        if (idle) {
            tile(step_idle);
            // (or the accumulators of the tile before would have to be kept for the way past this branch)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        } else {
            // the first fragments landed before the last barrier of the tile before (read there already, they would have to live through its
            // epilogue and through tiles without rows)
#pragma unroll
            for (int i = 0; i < 4; ++i) W[i] = frag(w_at + stage, i);
            X[0] = frag(x_at + stage, 0);
            X[1] = frag(x_at + stage, 1);
            read_scales(buffer_of(0), par, 0);
            CFP8_PHASE_END();
            // x tiles 2 and 3 of a tile's first step are added in its second
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i][2] = acc[i][3] = f32x4{0.f, 0.f, 0.f, 0.f};
            tile(step);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                add(i, 2, sc2[i & 1], false);
                add(i, 3, sc3[i & 1], false);
            }
        }

        if constexpr (DOWN) {
            // ---- bf16 rows.  A wave turns 16 of its rows at a time into stores of 128 contiguous bytes through the KiB of the last
            // step's stage that its own loads fill (every wave has read that stage before the step's barrier), and requests the
            // next tile's third step behind its last read.  16-byte piece c of row r at c ^ (r & 7).
            const int prev = stage == 0 ? 2 * STAGE : stage - STAGE;
            int le = lane;  // (addresses derived here: kept across the K loop they would cost registers)
            asm volatile("" : "+v"(le));
            const int lr = le & 15, lq = le >> 4;
            const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(p.out + (int64_t)m0 * p.N, 0, 0x80000000u, 0x00020000);
            uint8_t* const own = smem + prev + wave * 1024;
            const uint32_t turn = (uint32_t) reinterpret_cast<uintptr_t>((lds_void*)(own + (lr >> 3) * 8192 + (lr & 7) * 128 + (lq & 1) * 8));
            const uint8_t* const back = own + (le >> 3) * 128 + (((le & 7) ^ (le >> 3)) << 4);
            const uint32_t at = n0 + wn * 64 < p.N && !idle ? (uint32_t)((le >> 3) * p.N + n0 + wn * 64 + (le & 7) * 8) * 2u : kExOutside;
            // (LDS is written by instructions written out: in front of a store it knows of, the compiler waits for every load in flight)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int i = 0; i < 4 && !idle; ++i) {
                    const f32x4 v = acc[i][j];
                    const uint64_t two = (uint64_t)pack_bf16x2(v[0], v[1]) | ((uint64_t)pack_bf16x2(v[2], v[3]) << 32);
                    asm volatile("ds_write_b64 %0, %1 offset:%2" ::"v"(turn + (uint32_t)(((2 * i + (lq >> 1)) ^ (lr & 7)) << 4)), "v"(two), "n"((j & 1) * 16384) : "memory");
                }
                // written and read by one wave: its LDS operations complete in order
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const u32x4 d = *reinterpret_cast<const u32x4*>(back + (j & 1) * 16384 + r * 8192);
                    buffer_store16(d, ro, at, (uint32_t)(wm * 64 + j * 16 + r * 8) * (uint32_t)p.N * 2u);
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            dma_x(rxn, 2, prev, 0);
            dma_x(rxn, 2, prev, 1);
#pragma unroll
            for (int i = 0; i < 4; ++i) dma_w(rwn, 2, prev, i);
            CFP8_PHASE_END();
        } else {
            // ---- SwiGLU and quantisation.  Weight tiles 0 and 2 are gate rows, 1 and 3 the up rows of the same columns of h, so a lane
            // has both values of an element; both are rounded to bf16 first, as the product would be in memory.  A wave has 32 of the
            // 128 columns of the group: the four that share rows exchange their maxima.  Behind that a lane looks after one row (x tile
            // `quarter`, row lrow): its scale, and the 16 bytes of it that the four quarters hold a word of each.
            // A wave without rows stores nothing, or zeros and their scale for a down product that reads them.
            u32 h[2][4][2];  // [pair][x tile][two words of two bf16]
            int le = lane;  // (addresses derived here: kept across the K loop they would cost registers)
            asm volatile("" : "+v"(le));
            const int row = wm * 64 + le;  // x tile `quarter`, row lrow
            const uint32_t xch = (uint32_t) reinterpret_cast<uintptr_t>((lds_void*)(smem + kExExchange + row * 16));
            if (!idle) {
                u32 mx[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    u32 m = 0;
#pragma unroll
                    for (int pp = 0; pp < 2; ++pp) {
                        const f32x4 g = acc[2 * pp][j], u = acc[2 * pp + 1][j];
                        swiglu_quad(pack_bf16x2(g[0], g[1]), pack_bf16x2(g[2], g[3]), pack_bf16x2(u[0], u[1]), pack_bf16x2(u[2], u[3]), h[pp][j][0], h[pp][j][1]);
                        m = pk_absmax(pk_absmax(m, h[pp][j][0]), h[pp][j][1]);
                    }
                    mx[j] = pk_fold(m);
                }
                quarters_transpose(mx);  // the four quarters' maxima of row lrow of x tile `quarter`
                // (LDS by instructions written out: in front of a store it knows of, the compiler waits for every load in flight)
                asm volatile("ds_write_b32 %0, %1" ::"v"(xch + wn * 4), "v"(umax(umax(mx[0], mx[1]), umax(mx[2], mx[3]))) : "memory");
            }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            u32x4 bytes[2] = {u32x4{0u, 0u, 0u, 0u}, u32x4{0u, 0u, 0u, 0u}};
            float scale = scale_from_amax(0.f);
            if (!idle) {
                u32x4 all;
                asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(all) : "v"(xch) : "memory");
                scale = scale_from_amax(amax_from_bits(umax(umax(all[0], all[1]), umax(all[2], all[3]))));
                const Divider own(scale);
                u32 s4[4], r4[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s4[j] = __float_as_uint(own.s);
                    r4[j] = __float_as_uint(own.r);
                }
                quarters_transpose(s4);  // those of row lrow of x tile j
                quarters_transpose(r4);
#pragma unroll
                for (int pp = 0; pp < 2; ++pp) {
                    u32 q[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) q[j] = cast4(h[pp][j][0], h[pp][j][1], Divider(__uint_as_float(s4[j]), __uint_as_float(r4[j])));
                    quarters_transpose(q);
                    bytes[pp] = u32x4{q[0], q[1], q[2], q[3]};
                }
            }
            const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(p.h + (int64_t)m0 * (p.N >> 1), 0, 0x80000000u, 0x00020000);
            const __amdgpu_buffer_rsrc_t rh = __builtin_amdgcn_make_buffer_rsrc(p.hs + (int64_t)m0 * (p.N >> 8), 0, 0x80000000u, 0x00020000);
            const bool stores = !idle || p.whole_tiles;
#pragma unroll
            for (int pp = 0; pp < 2; ++pp) buffer_store16(bytes[pp], rq, stores ? (uint32_t)(row * (p.N >> 1)) : kExOutside, (uint32_t)((n0 >> 1) + wn * 32 + pp * 16));
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(scale), rh, wn == 0 && stores ? (uint32_t)(row * (p.N >> 8) * 4) : kExOutside, (uint32_t)((n0 >> 8) * 4), 0);
        }

        if (!has_next) break;
        pid = pid_n;
        m0 = m0n;
        n0 = n0n;
        rw = rwn;
        idle = wm == 1 && rows_n < kExBM;
        rx = rxn;
        rxs = rxsn;
        expert = expert_n;
        gb = buffer_of(G);
        par ^= 1;
    }
#undef CFP8_PRODUCT
    // the loads past the last tile land before the workgroup gives up its LDS
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// 4 to 32 K steps (the pipeline's depth and what one wave-wide load of weight scales covers), buffers that 32-bit offsets below
// kExOutside reach
bool experts_gate_up_takes(int64_t tokens, int64_t hidden, int64_t inter) {
    return hidden % 128 == 0 && hidden / 128 >= 4 && hidden / 128 <= 32 && inter % 128 == 0 && tokens * hidden <= 0xEFFFFFFFll && inter < (1 << 21);
}
bool experts_down_takes(int64_t hidden, int64_t inter) {
    return hidden % 128 == 0 && inter % 128 == 0 && inter / 128 >= 4 && inter / 128 <= 32 && hidden < (1 << 21);
}

template <bool DOWN, bool ONCE>
static int launch_experts(ExpertsArgs& p, int64_t rows, hipStream_t st) {
    p.tiles_m = (int)(rows / kExBM);
    p.tiles_n = (p.N + kExBN - 1) / kExBN;
    const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n;
    if (tiles > 0x7FFFFFFFll) return set_error(CFP8_EINVAL, "gemm: too many tiles for one launch");
    const int cus = cu_count();
    static std::atomic<bool> raised[65];  // zero-initialised
    const int slot = device_slot();
    if (slot == 64) raised[64].store(false, std::memory_order_relaxed);
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(gemm_experts_kernel<DOWN, ONCE>), kExLds, raised[slot])) return rc;
    const unsigned blocks = (unsigned)(tiles < cus ? tiles : cus);
    if (!note_launch(DOWN ? "gemm_experts<down>" : "gemm_experts<gate_up>", blocks, 512, kExLds)) return CFP8_OK;
    hipLaunchKernelGGL((gemm_experts_kernel<DOWN, ONCE>), dim3(blocks), dim3(512), kExLds, st, p);
    return check_launch("gemm");
}
// `once`: hardly an expert has a second tile of rows
int launch_experts_gate_up(ExpertsArgs& p, int64_t rows, bool once, hipStream_t st) { return once ? launch_experts<false, true>(p, rows, st) : launch_experts<false, false>(p, rows, st); }
int launch_experts_down(ExpertsArgs& p, int64_t rows, bool once, hipStream_t st) { return once ? launch_experts<true, true>(p, rows, st) : launch_experts<true, false>(p, rows, st); }

}  // namespace cfp8
