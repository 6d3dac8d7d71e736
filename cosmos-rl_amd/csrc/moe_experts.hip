// The experts of one MoE layer on routed tokens as one call: routing, 1x128 quantisation of the tokens, the gate_up product
// with SwiGLU, the down product and the weighted sum over each token's experts - launches only, on caller memory.
//
// Three forms, by the mean number of rows an expert gets:
//
//   many rows   Every expert's rows are padded to tiles of 128 (experts without a row get none).  The tokens are quantised
//               where they lie and gemm_experts_kernel gathers its rows from them; hidden sizes that it does not take are
//               quantised into the padded layout (cfp8_scatter_quant_group128) for the grouped GEMM of the training path.
//               Rows of padding: where a tile's second 64 rows are all padding and gemm_experts_kernel makes both products, those
//               rows of h are neither written nor read and hold what the workspace held (ExpertsArgs::whole_tiles).  All other
//               rows of padding are zeros all the way, which is what the grouped GEMMs of the training path are given. Rows past the last
//               group are not touched.
//   middle      A chunk of prefill: all experts' weights are read, for less than a tile of 128 rows each.  Rows lie one
//               behind the other without padding; the ring kernel takes tiles of 64 of one expert's rows (gemm_ring.hip:
//               kRingGateUp reads them from the quantised tokens and ends in SwiGLU, kRingDown), two workgroups a CU, or
//               down_stream_kernel the down weights strip by strip.  The
//               hidden activation is quantised in between, since a 1x128 group of it is spread over two workgroups.
//   few rows    A decode batch: reading the weights of the experts that have a row is all the time there is, and tiles of
//               64 rows would hold one or two.  One workgroup a CU, whose eight waves each take strips of 16 weight rows one
//               behind the other through LDS stages of their own, for tiles of 16 of an expert's rows (few_stream_kernel); with
//               less to read (few_streams) a workgroup takes a strip of ONE expert's weight rows, requests all of its K into
//               registers before anything else, and then walks the expert's rows in tiles of 16 (few_gate_up_kernel,
//               few_down_kernel).
#include <stdio.h>

#include <atomic>

#include "gemm_internal.h"
#include "moe_route.h"
#include "gemm_ring.h"

namespace cfp8 {

// few_gate_up_kernel and few_down_kernel hold a strip's whole K in registers: up to 8 K steps a wave of four (gate_up, 128 registers of weights and
// 64 of tokens), 12 a wave (down, 96 registers, and two tiles of 16 rows of 1536 bytes in LDS).  few_stream_kernel's tables of two tiles fit LDS beside
// its stages up to there (down 150 KiB), and its threads load one or two weight scales each and one activation scale (the static_asserts beside the loads).
constexpr int64_t kFewMaxHidden = 4096, kFewMaxInter = 1536;

struct FewArgs {
    const uint8_t* xq;       // [tokens, hidden] fp8
    const float* xs;         // [tokens, hidden / 128]
    const uint8_t* w;        // gate_up [experts, 2 inter, hidden] interleaved, or down [experts, hidden, inter]
    const float* ws;
    const int32_t* row_tokens;
    const int32_t* sizes;    // rows of every expert, and their inclusive cumulative sum
    const int32_t* ends;
    uint16_t* h;             // [rows, inter] bf16
    uint16_t* out;           // [rows, hidden] bf16
    int experts, hidden, inter, tokens;
};

// The slot-th expert that has rows (-1: there are fewer), and its rows.
__device__ __forceinline__ int few_expert(const FewArgs& p, int slot, int lane, int& start, int& end) {
    for (int e0 = 0; e0 < p.experts; e0 += 64) {
        const int n = e0 + lane < p.experts ? p.sizes[e0 + lane] : 0;
        const uint64_t has = __ballot(n > 0);
        const int c = __popcll(has);
        if (slot < c) {
            const uint64_t mine = __ballot(n > 0 && __popcll(has & ((1ull << lane) - 1)) == slot);
            const int bit = __ffsll((unsigned long long)mine) - 1;
            end = p.ends[e0 + bit];
            start = end - __builtin_amdgcn_readlane(n, bit);
            return e0 + bit;
        }
        slot -= c;
    }
    return -1;
}

__device__ __forceinline__ i32x8 few_frag(const u32x4& lo, const u32x4& hi) {
    return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
}

// ---------------------------------------------------------------------------
// gate_up and SwiGLU.  A workgroup of four waves: 16 gate rows and the 16 up rows of the same features (neighbours in the
// interleaved weight); wave w takes K steps w, w + 4, ... (NI of them), all of whose weights it requests at once.  Results
// have the bits of the grouped GEMMs: a lane reads bytes 32 q .. 32 q + 31 of a K step (q = lane >> 4) of both operands, as
// their fragments have them, and the steps' products meet in LDS unscaled, 16 steps a phase, from where one wave scales and
// adds them in the order of K.  h = bf16(bf16(silu(gate)) * up) leaves as bf16, since a 1x128 group of it is spread over
// eight workgroups.
// Bound by the weights' way in.  Whole calls, 128 experts of 2048 x 768, top 8, us: 16 tokens 95.5, 64 130.3 (91.5 and 126.6
// with loads of 64 contiguous bytes and every wave's own sum, which moves roundings: 2 of the 4 us are the loads).
// Cacheable against streaming loads, in both kernels: 16 tokens 96.2 / 102.0 behind kernels that write little, 143 / 106 behind
// one that left L2 full of its output; 64 tokens 131.6 / 141.7 and 180 / 147; 16 tokens on 4096 x 1536 282 / 310 and 326 / 316.
// Cacheable, since what runs in front of a decode batch's experts writes a few hundred kilobytes.
// ---------------------------------------------------------------------------
template <int NI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NI <= 4 ? 4 : 2))) void few_gate_up_kernel(const FewArgs p) {
    __shared__ __attribute__((aligned(16))) f32x4 prod[16][2][64];
    __shared__ float factor[16][2][16];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lrow = lane & 15, quarter = lane >> 4;
    const int KT = p.hidden >> 7, strip = blockIdx.x;
    int start, end;
    const int e = few_expert(p, (int)blockIdx.y, lane, start, end);
    if (e < 0) return;
    const uint8_t* const wg = p.w + ((int64_t)e * 2 * p.inter + strip * 32 + lrow) * p.hidden + quarter * 32;
    const uint8_t* const wu = wg + (int64_t)16 * p.hidden;
    u32x4 w[NI][4];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int kt = wave + 4 * i < KT ? wave + 4 * i : KT - 1;
        w[i][0] = *reinterpret_cast<const u32x4*>(wg + (kt << 7));
        w[i][1] = *reinterpret_cast<const u32x4*>(wg + (kt << 7) + 16);
        w[i][2] = *reinterpret_cast<const u32x4*>(wu + (kt << 7));
        w[i][3] = *reinterpret_cast<const u32x4*>(wu + (kt << 7) + 16);
    }
    float sg[NI], su[NI];
    const float* const sp = p.ws + ((int64_t)e * (p.inter >> 6) + 2 * (strip >> 3)) * KT;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int kt = wave + 4 * i < KT ? wave + 4 * i : KT - 1;
        sg[i] = sp[kt];
        su[i] = sp[KT + kt];
    }
    for (int r0 = start; r0 < end; r0 += 16) {
        const int row = r0 + lrow;
        const int64_t token = p.row_tokens[row < end ? row : end - 1];
        const uint8_t* const xp = p.xq + token * p.hidden + quarter * 32;
        const float* const xsp = p.xs + token * KT;
        u32x4 x[NI][2];
        float xs[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int kt = wave + 4 * i < KT ? wave + 4 * i : KT - 1;
            x[i][0] = *reinterpret_cast<const u32x4*>(xp + (kt << 7));
            x[i][1] = *reinterpret_cast<const u32x4*>(xp + (kt << 7) + 16);
            xs[i] = xsp[kt];
        }
        const bool adds = wave == ((r0 - start) >> 4 & 3) && row < end;  // the tiles' sums are taken in turn
        f32x4 g = {0.f, 0.f, 0.f, 0.f}, u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ph = 0; ph < (NI + 3) / 4; ++ph) {
            if (ph || r0 != start) __syncthreads();  // the sums of the phase before have been taken
#pragma unroll
            for (int i = 4 * ph; i < NI && i < 4 * ph + 4; ++i) {
                if (i == NI - 1 && wave + 4 * i >= KT) continue;
                const i32x8 xf = few_frag(x[i][0], x[i][1]);
                const f32x4 pg = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(few_frag(w[i][0], w[i][1]), xf, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
                const f32x4 pu = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(few_frag(w[i][2], w[i][3]), xf, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
                const int at = wave + 4 * (i - 4 * ph);
                if (row < end) {
                    prod[at][0][lane] = pg;
                    prod[at][1][lane] = pu;
                    if (quarter == 0) {
                        factor[at][0][lrow] = xs[i] * sg[i];
                        factor[at][1][lrow] = xs[i] * su[i];
                    }
                }
            }
            __syncthreads();
            if (adds) {
                const int steps = KT - 16 * ph < 16 ? KT - 16 * ph : 16;
#pragma unroll 4
                for (int s = 0; s < steps; ++s) {
                    const f32x4 pg = prod[s][0][lane], pu = prod[s][1][lane];
                    const float fg = factor[s][0][lrow], fu = factor[s][1][lrow];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        g[k] = __builtin_fmaf(pg[k], fg, g[k]);
                        u[k] = __builtin_fmaf(pu[k], fu, u[k]);
                    }
                }
            }
        }
        if (adds) {
            u32 h0, h1;
            swiglu_quad(pack_bf16x2(g[0], g[1]), pack_bf16x2(g[2], g[3]), pack_bf16x2(u[0], u[1]), pack_bf16x2(u[2], u[3]), h0, h1);
            *reinterpret_cast<uint2*>(p.h + (int64_t)row * p.inter + strip * 16 + quarter * 4) = make_uint2(h0, h1);
        }
    }
}

// ---------------------------------------------------------------------------
// down.  A workgroup of eight waves: 128 weight rows, 16 a wave over the whole of K (NI = inter / 128 steps), all requested
// at once; under those loads the workgroup quantises 16 rows of h (1x128, as the quantiser does) into LDS.  About 27 us
// for the 129 MB of 16 tokens' experts (2048 x 768); the grouped GEMM on tiles of 128 rows took 68 us.
// ---------------------------------------------------------------------------
template <int NI>
__global__ __launch_bounds__(512) void few_down_kernel(const FewArgs p) {
    constexpr int PITCH = NI * 128 + 16;
    __shared__ __attribute__((aligned(16))) uint8_t q[2][16 * PITCH];
    __shared__ float qs[2][16][NI];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lrow = lane & 15, quarter = lane >> 4;
    int start, end;
    const int e = few_expert(p, (int)blockIdx.y, lane, start, end);
    if (e < 0) return;
    const int n0 = (int)blockIdx.x * 128 + wave * 16;
    const uint8_t* const wp = p.w + ((int64_t)e * p.hidden + n0 + lrow) * p.inter + quarter * 32;
    u32x4 w[NI][2];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        w[i][0] = *reinterpret_cast<const u32x4*>(wp + (i << 7));
        w[i][1] = *reinterpret_cast<const u32x4*>(wp + (i << 7) + 16);
    }
    float sw[NI];
    const float* const sp = p.ws + ((int64_t)e * (p.hidden >> 7) + blockIdx.x) * NI;
#pragma unroll
    for (int i = 0; i < NI; ++i) sw[i] = sp[i];
    int turn = 0;
    for (int r0 = start; r0 < end; r0 += 16, turn ^= 1) {
        const int rows = end - r0 < 16 ? end - r0 : 16;
        for (int g = t >> 4; g < rows * NI; g += 32) {
            const int r = g / NI, c = g - r * NI, sub = t & 15;
            const uint4 v = *reinterpret_cast<const uint4*>(p.h + (int64_t)(r0 + r) * p.inter + c * 128 + sub * 8);
            const float scale = scale_from_amax(amax_from_bits(row16_max(pk_fold(absmax8(0u, v)))));
            *reinterpret_cast<uint2*>(&q[turn][r * PITCH + c * 128 + sub * 8]) = cast8(v, Divider(scale));
            if (sub == 0) qs[turn][r][c] = scale;
        }
        __syncthreads();
        const int rr = lrow < rows ? lrow : rows - 1;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const u32x4 lo = *reinterpret_cast<const u32x4*>(&q[turn][rr * PITCH + i * 128 + quarter * 32]);
            const u32x4 hi = *reinterpret_cast<const u32x4*>(&q[turn][rr * PITCH + i * 128 + quarter * 32 + 16]);
            const f32x4 pr = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(few_frag(w[i][0], w[i][1]), few_frag(lo, hi), f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
            const float f = qs[turn][rr][i] * sw[i];
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[k] = __builtin_fmaf(pr[k], f, acc[k]);
        }
        if (lrow < rows)
            *reinterpret_cast<uint2*>(p.out + (int64_t)(r0 + lrow) * p.hidden + n0 + quarter * 4) =
                make_uint2(pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]));
    }
}

// ---------------------------------------------------------------------------
// The same two products with one workgroup of eight waves a CU, every wave a stream of strips.  Units are (tile of 16 of an expert's rows, strip of 16 weight
// rows), numbered tile by tile; a workgroup takes an even share of them, which lies in one or two tiles (there are no more tiles than
// workgroups), its waves every eighth.  A wave has all of K of its strip, step by step through LDS stages of its own, and the loads run on from unit to
// unit; products are scaled and added in the order of K, with the bits of the kernels above.  No barrier behind the workgroup's tables of its two tiles.
//
// Bound by the weights' way in: as a stream alone (258 MB) 8 rows x 128 bytes a load into LDS take 39.6 us, 32 bytes a lane of sixteen rows, which the kernels above
// request, 45.8.  16 tokens, top 8 of 128 experts of 2048 x 768: gate_up 53 -> 45 us, down 27 -> 23; the four waves' worth of steps at a workgroup's end and 2 us of tables are
// the rest.  Streaming loads: cacheable ones 45 -> 53 us and the call 81 -> 91.
// ---------------------------------------------------------------------------
constexpr uint32_t kFewOutside = 0xF0000000u;  // a per-lane offset past the end of every buffer
constexpr int kStreamWaves = 8;
constexpr int kStreamMostExperts = 256;        // four a lane

// inclusive sums over the lanes: within sixteen, then the lasts of sixteen into the next and of 32 into the upper half (by shuffles, 24 of them in a chain, 1.5 us a kernel)
__device__ __forceinline__ u32 wave_sums(u32 x) {
    int v = (int)x;
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);
    return (u32)v;
}

struct StreamTile {
    int expert, row, rows;  // rows 1 .. ROWS
};

// Tiles of ROWS rows of all experts, expert by expert: lane l of group g has expert 64 g + l, its tiles and rows up to and with it in the halves of a word.
template <int ROWS>
struct StreamTiles {
    u32 upto[kStreamMostExperts / 64], own[kStreamMostExperts / 64];
    int total;
    __device__ __forceinline__ StreamTiles(const int32_t* sizes, int experts, int lane) {
        u32 before = 0;
#pragma unroll
        for (int g = 0; g < kStreamMostExperts / 64; ++g) own[g] = g * 64 + lane < experts ? (u32)sizes[g * 64 + lane] : 0u;
#pragma unroll
        for (int g = 0; g < kStreamMostExperts / 64; ++g) {
            own[g] |= ((own[g] + (ROWS - 1u)) / ROWS) << 16;
            upto[g] = before + (g * 64 < experts ? wave_sums(own[g]) : 0u);
            before = (u32)__builtin_amdgcn_readlane((int)upto[g], 63);
        }
        total = (int)(before >> 16);
    }
    __device__ __forceinline__ StreamTile find(int tile) const {  // tile < total
        StreamTile t{0, 0, 0};
#pragma unroll
        for (int g = kStreamMostExperts / 64 - 1; g >= 0; --g) {
            const uint64_t past = __ballot((int)(upto[g] >> 16) > tile);
            if (!past) break;
            const int bit = __ffsll((unsigned long long)past) - 1;
            const u32 end = (u32)__builtin_amdgcn_readlane((int)upto[g], bit), mine = (u32)__builtin_amdgcn_readlane((int)own[g], bit);
            const int at = tile - (int)((end >> 16) - (mine >> 16)), left = (int)(mine & 0xFFFFu) - at * ROWS;
            t = {g * 64 + bit, (int)((end & 0xFFFFu) - (mine & 0xFFFFu)) + at * ROWS, left < ROWS ? left : ROWS};
        }
        return t;
    }
};

// D: stages of a wave
template <bool DOWN, int D>
__global__ __launch_bounds__(kStreamWaves * 64) void few_stream_kernel(const FewArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    typedef __attribute__((address_space(3))) void lds_void;
    constexpr int STAGE = DOWN ? 2048 : 4096, L = DOWN ? 2 : 4;  // bytes and loads of a step: gate_up takes its rows of the tokens as well
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lrow = lane & 15, quarter = lane >> 4;
    const int K = DOWN ? p.inter : p.hidden, KT = K >> 7, pitch = KT | 1;
    const int N = DOWN ? p.hidden : 2 * p.inter, strips = N >> 4;
    const StreamTiles<16> tiles(p.sizes, p.experts, lane);
    const int64_t units = (int64_t)tiles.total * strips;
    const int first = (int)(units * blockIdx.x / gridDim.x), end = (int)(units * (blockIdx.x + 1) / gridDim.x);
    if (first >= end) return;
    const int tile0 = first / strips, change = (tile0 + 1) * strips;  // from unit `change` on the second tile
    const bool two = end > change;
    const StreamTile ta = tiles.find(tile0), tb = two ? tiles.find(tile0 + 1) : ta;

    // ---- tables of the two tiles: down: rows of h, quantised, as stages [K step][16][128]; activation scales [16][pitch], weight scales [N / 128][KT]
    const int sa_words = 16 * pitch, sb_words = (N >> 7) * KT, q_bytes = DOWN ? KT * 2048 : 0;
    const int table = (q_bytes + (sa_words + sb_words) * 4 + 255) & ~255;
    uint8_t* const own = smem + 2 * table + wave * D * STAGE;

    const uint32_t wbytes = (uint32_t)N * (uint32_t)K;
    const uint8_t* const wa = p.w + (uint64_t)ta.expert * wbytes;
    const uint8_t* const wb = p.w + (uint64_t)tb.expert * wbytes;
    const __amdgpu_buffer_rsrc_t rwa = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(wa), 0, (int)wbytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rwb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(wb), 0, (int)wbytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.xq), 0, DOWN ? 0 : (int)((uint32_t)p.tokens * (uint32_t)K), 0x00020000);
    // a load of 8 rows x 128 bytes: row lane >> 3, whose 16-byte chunk c lies at position c ^ f(row), f(row) = bit 1 of row | (bit 3 of row) << 2
    auto chunk_of = [&](int half) { return (uint32_t)((lane & 7) ^ (((lane >> 4) & 1) | (half << 2))) * 16u; };
    const uint32_t vw[2] = {(uint32_t)(lane >> 3) * (uint32_t)K + chunk_of(0), (uint32_t)(lane >> 3) * (uint32_t)K + chunk_of(1)};

    // rows of the tokens that the lanes load, in front of the weights: these do not wait for them
    int token[2][2] = {{-1, -1}, {-1, -1}};
    int srow[2] = {-1, -1};  // the token of row t >> 5 of a tile, for the tables
    if constexpr (!DOWN) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = h * 8 + (lane >> 3);
            if (r < ta.rows) token[0][h] = p.row_tokens[ta.row + r];
            if (two && r < tb.rows) token[1][h] = p.row_tokens[tb.row + r];
        }
        if ((t >> 5) < ta.rows) srow[0] = p.row_tokens[ta.row + (t >> 5)];
        if (two && (t >> 5) < tb.rows) srow[1] = p.row_tokens[tb.row + (t >> 5)];
    }
    // ---- the stream of loads: unit iu, step ik
    int iu = first + wave, ik = 0;
    auto strip_row = [&](int u) {  // the strip's first weight row; gate_up: 8 gate rows, and the up rows of the same features 16 behind them
        const int s = u - (u >= change ? change : change - strips);
        return DOWN ? s * 16 : (s >> 1) * 32 + (s & 1) * 8;
    };
    uint32_t ibase = (uint32_t)strip_row(iu) * (uint32_t)K;
    uint32_t vx[2][2];
    auto load_w = [&](int st) {
        const bool in = iu < end, b = iu >= change;
        uint8_t* const to = own + st * STAGE;
        const uint32_t at = ibase + ((uint32_t)ik << 7), second = at + (DOWN ? 8u : 16u) * (uint32_t)K;
        const __amdgpu_buffer_rsrc_t r = b ? rwb : rwa;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)to, 16, in ? vw[0] : kFewOutside, at, 0, 2);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)(to + 1024), 16, in ? vw[1] : kFewOutside, second, 0, 2);
    };
    auto load_x = [&](int st) {
        const bool in = iu < end, b = iu >= change;
        uint8_t* const to = own + st * STAGE + 2048;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint8_t* const half = to + h * 1024;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void*)half, 16, !in ? kFewOutside : b ? vx[1][h] : vx[0][h], (uint32_t)ik << 7, 0, 0);
        }
    };
    auto advance = [&]() {
        if (++ik == KT) {
            ik = 0;
            iu += kStreamWaves;
            ibase = (uint32_t)strip_row(iu < end ? iu : first) * (uint32_t)K;
        }
    };

    if constexpr (DOWN) {
        // h in front of the weights; 16 lanes a group of 128, 32 groups at a time
        const int groups = (ta.rows + (two ? tb.rows : 0)) * KT;
        uint4 v[3];
        auto group_of = [&](int g, int& r, int& c, bool& second) {
            const int row = g / KT;
            c = g - row * KT;
            second = row >= ta.rows;
            r = second ? row - ta.rows : row;
        };
        auto fetch = [&](int g) {
            int r, c;
            bool second;
            group_of(g, r, c, second);
            return *reinterpret_cast<const uint4*>(p.h + (int64_t)((second ? tb.row : ta.row) + r) * K + c * 128 + (t & 15) * 8);
        };
        auto store = [&](int g, const uint4& d) {
            int r, c;
            bool second;
            group_of(g, r, c, second);
            const float scale = scale_from_amax(amax_from_bits(row16_max(pk_fold(absmax8(0u, d)))));
            const uint2 q = cast8(d, Divider(scale));
            const int ch = ((t & 15) >> 1) ^ (((r >> 1) & 1) | (((r >> 3) & 1) << 2));
            uint8_t* const tab = smem + (second ? table : 0);
            const uint32_t at = (uint32_t) reinterpret_cast<uintptr_t>((lds_void*)(tab + c * 2048 + r * 128 + ch * 16 + (t & 1) * 8));
            const uint64_t two_words = (uint64_t)q.x | ((uint64_t)q.y << 32);
            // (LDS by instructions written out: in front of a store it knows of, the compiler waits for every load in flight)
            asm volatile("ds_write_b64 %0, %1" ::"v"(at), "v"(two_words) : "memory");
            if ((t & 15) == 0) {
                const uint32_t sat = (uint32_t) reinterpret_cast<uintptr_t>((lds_void*)(tab + q_bytes + (r * pitch + c) * 4));
                asm volatile("ds_write_b32 %0, %1" ::"v"(sat), "v"(scale) : "memory");
            }
        };
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int g = i * 32 + (t >> 4);
            if (g < groups) v[i] = fetch(g);
        }
        static_assert(kFewMaxHidden / 128 * (kFewMaxInter / 128) <= kStreamWaves * 64, "a weight scale a thread");
        float sw[2];
#pragma unroll
        for (int b = 0; b < 2; ++b)
            if (t < sb_words) sw[b] = p.ws[(int64_t)(b ? tb.expert : ta.expert) * sb_words + t];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            load_w(d);
            advance();
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const uint32_t at = (uint32_t) reinterpret_cast<uintptr_t>((lds_void*)(smem + b * table + q_bytes + (sa_words + t) * 4));
            if (t < sb_words) asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(sw[b]) : "memory");
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int g = i * 32 + (t >> 4);
            if (g < groups) store(g, v[i]);
        }
        for (int g = 96 + (t >> 4); g < groups; g += 32) store(g, fetch(g));
    } else {
        // what needs no token, the weights, then what the tokens' numbers were waited for
        static_assert(2 * kFewMaxInter / 128 * (kFewMaxHidden / 128) <= 2 * kStreamWaves * 64 && kFewMaxHidden / 128 <= 32, "two weight scales a thread, an activation scale");
        float sw[2][2], sx[2];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                if (t + i * kStreamWaves * 64 < sb_words) sw[b][i] = p.ws[(int64_t)(b ? tb.expert : ta.expert) * sb_words + t + i * kStreamWaves * 64];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            load_w(d);
            advance();
        }
        iu = first + wave;
        ik = 0;
        ibase = (uint32_t)strip_row(iu < end ? iu : first) * (uint32_t)K;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int tok = srow[b];
            sx[b] = 0.f;
            if (tok >= 0 && (t & 31) < KT) sx[b] = p.xs[(int64_t)tok * KT + (t & 31)];
#pragma unroll
            for (int h = 0; h < 2; ++h) vx[b][h] = token[b][h] >= 0 ? (uint32_t)token[b][h] * (uint32_t)K + chunk_of(h) : kFewOutside;
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            load_x(d);
            advance();
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            uint8_t* const tab = smem + b * table;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t at = (uint32_t) reinterpret_cast<uintptr_t>((lds_void*)(tab + (sa_words + t + i * kStreamWaves * 64) * 4));
                if (t + i * kStreamWaves * 64 < sb_words) asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(sw[b][i]) : "memory");
            }
            const uint32_t at = (uint32_t) reinterpret_cast<uintptr_t>((lds_void*)(tab + ((t >> 5) * pitch + (t & 31)) * 4));
            if ((t & 31) < KT) asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(sx[b]) : "memory");
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    const int fr = ((lrow >> 1) & 1) | (((lrow >> 3) & 1) << 2);
    const int fo = lrow * 128 + (((2 * quarter) ^ fr) << 4);
    auto frag = [&](const uint8_t* at) {
        const i32x4 lo = *reinterpret_cast<const i32x4*>(at + fo);
        const i32x4 hi = *reinterpret_cast<const i32x4*>(at + (fo ^ 16));
        return i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    int st = 0;
    int fresh = DOWN ? 0 : D;  // gate_up's first steps: their rows of the tokens were requested behind all their weights
    for (int u = first + wave; u < end; u += kStreamWaves) {
        const bool b = u >= change;
        const uint8_t* const tab = smem + (b ? table : 0);
        const int row0 = strip_row(u), s = u - (b ? change : change - strips);
        const float* const sa = reinterpret_cast<const float*>(tab + q_bytes) + lrow * pitch;
        // gate_up: gate scales for lanes of gate rows, up scales for the others; down: the strip's block
        const float* const sb = reinterpret_cast<const float*>(tab + q_bytes) + sa_words + (DOWN ? s >> 3 : (s >> 4) * 2 + (quarter >> 1)) * KT;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < KT; ++k) {
            if (!DOWN && fresh > 0) {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (D - 1)) : "memory");
                --fresh;
            } else {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L * (D - 1)) : "memory");
            }
            const uint8_t* const at = own + st * STAGE;
            const i32x8 w = frag(at), x = frag(DOWN ? tab + k * 2048 : at + 2048);
            const float f = sa[k] * sb[k];
            const f32x4 pr = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, x, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(pr[e], f, acc[e]);
            asm volatile("" : "+v"(acc));  // the fragments have been read
            __builtin_amdgcn_sched_barrier(0);
            load_w(st);
            if constexpr (!DOWN) load_x(st);
            advance();
            st = st == D - 1 ? 0 : st + 1;
        }
        const int row = (b ? tb.row : ta.row) + lrow;
        const bool stores = lrow < (b ? tb.rows : ta.rows);
        const u32 p0 = pack_bf16x2(acc[0], acc[1]), p1 = pack_bf16x2(acc[2], acc[3]);
        if constexpr (DOWN) {
            if (stores) *reinterpret_cast<uint2*>(p.out + (int64_t)row * N + row0 + quarter * 4) = make_uint2(p0, p1);
        } else {
            // quarters 0 and 1 have the gate rows, 2 and 3 the up rows of the same features
            const u32 u0 = __builtin_amdgcn_permlane32_swap(p0, p0, false, false)[1], u1 = __builtin_amdgcn_permlane32_swap(p1, p1, false, false)[1];
            u32 h0, h1;
            swiglu_quad(p0, p1, u0, u1, h0, h1);
            if (stores && quarter < 2) *reinterpret_cast<uint2*>(p.h + (int64_t)row * p.inter + s * 8 + quarter * 4) = make_uint2(h0, h1);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may land in LDS once the workgroup has gone
}

template <bool DOWN>
static int launch_few_stream(const FewArgs& p, hipStream_t st) {
    constexpr int D = DOWN ? 6 : 4;  // (3 and 4 level; 6 and 4 within 1 %)
    const int K = DOWN ? p.inter : p.hidden, N = DOWN ? p.hidden : 2 * p.inter, KT = K / 128;
    const size_t table = ((DOWN ? KT * 2048 : 0) + (16 * (KT | 1) + N / 128 * KT) * 4 + 255) & ~255;
    const size_t lds = 2 * table + (size_t)kStreamWaves * D * (DOWN ? 2048 : 4096);
    static std::atomic<bool> raised[65];
    const int slot = device_slot();
    if (slot == 64) raised[64].store(false, std::memory_order_relaxed);
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(few_stream_kernel<DOWN, D>), 160 * 1024, raised[slot])) return rc;
    hipLaunchKernelGGL((few_stream_kernel<DOWN, D>), dim3((unsigned)cu_count()), dim3(kStreamWaves * 64), lds, st, p);
    return check_launch("moe_experts");
}

// ---------------------------------------------------------------------------
// down of the middle form: the same stream of weights for tiles of 16 TM rows, already quantised, of which the workgroup keeps its one or two in LDS whole ([K
// step][16 rows][128 bytes]).  A store is issued for every 16 rows of a tile, whether it has them or not (what lies behind the tile is dropped): for D steps the waits
// for loads count the stores behind them.
// Bound by the weights' way in and the stores: 201 MB (128 experts of 2048 x 768), 13 rows an expert 47 -> 37 us (5.4 TB/s), 28: 50 -> 42, where the ring kernel's tiles of
// 64 x 128 load their rows for every 128 columns and fill and drain their rings for six K steps.  D = 3 and 5 are level.
// ---------------------------------------------------------------------------
struct DownArgs {
    const uint8_t* hq;     // [rows, inter] fp8
    const float* hs;       // [rows, inter / 128]
    const uint8_t* w;      // [experts, hidden, inter]
    const float* ws;
    const int32_t* sizes;  // rows of every expert, which lie one behind the other
    uint16_t* out;         // [rows, hidden] bf16
    int experts, hidden, inter;
};

template <int TM, int D>
__global__ __launch_bounds__(kStreamWaves * 64) void down_stream_kernel(const DownArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    typedef __attribute__((address_space(3))) void lds_void;
    constexpr int ROWS = TM * 16, STAGE = 2048, L = 2;
    static_assert(ROWS <= 64, "a lane a row");
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lrow = lane & 15, quarter = lane >> 4;
    const int K = p.inter, KT = K >> 7, pitch = KT | 1, N = p.hidden, strips = N >> 4;
    const StreamTiles<ROWS> tiles(p.sizes, p.experts, lane);
    const int64_t units = (int64_t)tiles.total * strips;
    const int first = (int)(units * blockIdx.x / gridDim.x), end = (int)(units * (blockIdx.x + 1) / gridDim.x);
    if (first >= end) return;
    const int tile0 = first / strips, change = (tile0 + 1) * strips;  // from unit `change` on the second tile
    const bool two = end > change;
    const StreamTile ta = tiles.find(tile0), tb = two ? tiles.find(tile0 + 1) : ta;

    // ---- tables of the two tiles: rows of h, activation scales [ROWS][pitch], weight scales [N / 128][KT]
    const int sa_words = ROWS * pitch, sb_words = (N >> 7) * KT, q_bytes = KT * ROWS * 128;
    const int table = (q_bytes + (sa_words + sb_words) * 4 + 255) & ~255;
    uint8_t* const own = smem + 2 * table + wave * D * STAGE;
    const uint32_t wbytes = (uint32_t)N * (uint32_t)K;
    auto tile_rsrc = [&](const void* base, int64_t row, int rows, int row_bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(static_cast<uint8_t*>(const_cast<void*>(base)) + row * row_bytes, 0, rows * row_bytes, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rwa = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w) + (uint64_t)ta.expert * wbytes, 0, (int)wbytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rwb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w) + (uint64_t)tb.expert * wbytes, 0, (int)wbytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t roa = tile_rsrc(p.out, ta.row, ta.rows, N * 2), rob = tile_rsrc(p.out, tb.row, tb.rows, N * 2);
    // (few_stream_kernel's order of a row's chunks)
    auto chunk_of = [&](int half) { return (uint32_t)((lane & 7) ^ (((lane >> 4) & 1) | (half << 2))) * 16u; };
    const uint32_t vw[2] = {(uint32_t)(lane >> 3) * (uint32_t)K + chunk_of(0), (uint32_t)(lane >> 3) * (uint32_t)K + chunk_of(1)};

    for (int b = 0; b < (two ? 2 : 1); ++b) {
        const __amdgpu_buffer_rsrc_t rx = b ? tile_rsrc(p.hq, tb.row, tb.rows, K) : tile_rsrc(p.hq, ta.row, ta.rows, K);
        for (int l = wave; l < KT * 2 * TM; l += kStreamWaves) {
            const int j = l / (2 * TM), g = l - j * 2 * TM;
            uint8_t* const to = smem + b * table + l * 1024;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void*)to, 16, (uint32_t)(g >> 1) * 16u * (uint32_t)K + ((g & 1) ? vw[1] + 8u * (uint32_t)K : vw[0]), (uint32_t)j << 7, 0, 0);
        }
    }
    float sw[2], sx[2] = {0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const StreamTile& tile = b ? tb : ta;
        if (t < sb_words) sw[b] = p.ws[(int64_t)tile.expert * sb_words + t];
        if (t < tile.rows * KT) sx[b] = p.hs[(int64_t)tile.row * KT + t];
    }
    // ---- the stream of loads: unit iu, step ik
    int iu = first + wave, ik = 0;
    auto strip_of = [&](int u) { return u - (u >= change ? change : change - strips); };
    uint32_t ibase = (uint32_t)strip_of(iu) * 16u * (uint32_t)K;
    auto load_w = [&](int st) {
        const bool in = iu < end;
        uint8_t* const to = own + st * STAGE;
        const uint32_t at = ibase + ((uint32_t)ik << 7);
        const __amdgpu_buffer_rsrc_t r = iu >= change ? rwb : rwa;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)to, 16, in ? vw[0] : kFewOutside, at, 0, 2);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)(to + 1024), 16, in ? vw[1] : kFewOutside, at + 8u * (uint32_t)K, 0, 2);
        if (++ik == KT) {
            ik = 0;
            iu += kStreamWaves;
            ibase = (uint32_t)strip_of(iu < end ? iu : first) * 16u * (uint32_t)K;
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load_w(d);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int r = t / KT, c = t - r * KT;
        const uint32_t base = (uint32_t) reinterpret_cast<uintptr_t>((lds_void*)(smem + b * table + q_bytes));
        if (t < ROWS * KT) asm volatile("ds_write_b32 %0, %1" ::"v"(base + (uint32_t)(r * pitch + c) * 4u), "v"(sx[b]) : "memory");
        if (t < sb_words) asm volatile("ds_write_b32 %0, %1" ::"v"(base + (uint32_t)(sa_words + t) * 4u), "v"(sw[b]) : "memory");
    }
    // the tables are older than the weights' first stages
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(L * D) : "memory");

    const int fr = ((lrow >> 1) & 1) | (((lrow >> 3) & 1) << 2);
    const int fo = lrow * 128 + (((2 * quarter) ^ fr) << 4);
    auto frag = [&](const uint8_t* at) {
        const i32x4 lo = *reinterpret_cast<const i32x4*>(at + fo);
        const i32x4 hi = *reinterpret_cast<const i32x4*>(at + (fo ^ 16));
        return i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    int st = 0, stored = 0;  // steps left whose loads are older than the last stores
    for (int u = first + wave; u < end; u += kStreamWaves) {
        const bool b = u >= change;
        const uint8_t* const tab = smem + (b ? table : 0);
        const int s = strip_of(u);
        const float* const sa = reinterpret_cast<const float*>(tab + q_bytes) + lrow * pitch;
        const float* const sb = reinterpret_cast<const float*>(tab + q_bytes) + sa_words + (s >> 3) * KT;
        f32x4 acc[TM];
#pragma unroll
        for (int m = 0; m < TM; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < KT; ++k) {
            if (stored > 0) {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L * (D - 1) + TM) : "memory");
                --stored;
            } else {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L * (D - 1)) : "memory");
            }
            const i32x8 w = frag(own + st * STAGE);
            const float f = sb[k];
#pragma unroll
            for (int m = 0; m < TM; ++m) {
                const i32x8 x = frag(tab + (k * TM + m) * 2048);
                const float fm = sa[m * 16 * pitch + k] * f;
                const f32x4 pr = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, x, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[m][e] = __builtin_fmaf(pr[e], fm, acc[m][e]);
            }
#pragma unroll
            for (int m = 0; m < TM; ++m) asm volatile("" : "+v"(acc[m]));  // the fragments have been read
            __builtin_amdgcn_sched_barrier(0);
            load_w(st);
            st = st == D - 1 ? 0 : st + 1;
        }
        const __amdgpu_buffer_rsrc_t ro = b ? rob : roa;
#pragma unroll
        for (int m = 0; m < TM; ++m)
            __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack_bf16x2(acc[m][0], acc[m][1]), pack_bf16x2(acc[m][2], acc[m][3])}, ro,
                                                  (uint32_t)(m * 16 + lrow) * (uint32_t)N * 2u + (uint32_t)quarter * 8u, (uint32_t)s * 32u, 0);
        stored = D;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may land in LDS once the workgroup has gone
}

constexpr int kDownStreamDepth = 3;
static size_t down_stream_lds(int64_t hidden, int64_t inter, int rows) {
    const int64_t KT = inter / 128;
    return (size_t)(2 * ((KT * rows * 128 + (rows * (KT | 1) + hidden / 128 * KT) * 4 + 255) & ~(int64_t)255) + kStreamWaves * kDownStreamDepth * 2048);
}
// Rows of a tile of down_stream_kernel in the middle form, 0: the ring kernel is taken.  The most rows of which LDS holds two tiles; fewer are level where an expert seldom has more
// (13 and 20 rows an expert, tiles of 64, 48 and 32: 121, 121, 121 and 127, 127, 126 us a call) and behind where it has (36: 138.5, 139.8, 145.9).  Up to three
// quarters of a tile an expert, beyond which second tiles read the weights again; no more tiles than workgroups, and weights of 32 MiB and more.  Whole calls, us, ring / streams, 128 experts of 2048 x 768, top 8: 13
// rows 129.7 / 121.2, 28: 140.4 / 131.7, 42: 149.3 / 142.6; of 3584 x 640: 32: 202 / 191; 64 of 1024 x 512, top 6: 13: 36.1 / 35.9, 40: 43.1 / 43.0; 64 of 2048 x 1024, top 8 (48 rows): 20: 91.3 /
// 88.0, 36: 97.2 / 97.0, 48: 101.9 / 108.9; 32 of 3584 x 1536, top 4 (32 rows): 16: 113.3 / 108.7, 24: 115.4 / 113.3, 30: 114.4 / 119.7.
static int down_stream_rows(int64_t pairs, int64_t slots, int64_t experts, int64_t hidden, int64_t inter) {
    const int64_t KT = inter / 128;
    if (experts > kStreamMostExperts || hidden / 128 * KT > kStreamWaves * 64 || slots * hidden * inter < (int64_t)32 << 20) return 0;
    for (int rows = 64; rows >= 32; rows -= 16)
        if (rows * KT <= kStreamWaves * 64 && down_stream_lds(hidden, inter, rows) <= 160 * 1024)
            return slots + pairs / rows <= cu_count() && pairs <= rows * 3 / 4 * experts ? rows : 0;
    return 0;
}
template <int TM>
static int launch_down_stream(const DownArgs& p, hipStream_t st) {
    auto* const kern = down_stream_kernel<TM, kDownStreamDepth>;
    static std::atomic<bool> raised[65];
    const int slot = device_slot();
    if (slot == 64) raised[64].store(false, std::memory_order_relaxed);
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kern), 160 * 1024, raised[slot])) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)cu_count()), dim3(kStreamWaves * 64), down_stream_lds(p.hidden, p.inter, TM * 16), st, p);
    return check_launch("moe_experts");
}

template <int NI>
static void launch_few_gate_up(int ni, dim3 grid, hipStream_t st, const FewArgs& p) {
    if constexpr (NI > 0) {
        if (ni == NI) hipLaunchKernelGGL(few_gate_up_kernel<NI>, grid, dim3(256), 0, st, p);
        else launch_few_gate_up<NI - 1>(ni, grid, st, p);
    }
}
template <int NI>
static void launch_few_down(int ni, dim3 grid, hipStream_t st, const FewArgs& p) {
    if constexpr (NI > 0) {
        if (ni == NI) hipLaunchKernelGGL(few_down_kernel<NI>, grid, dim3(512), 0, st, p);
        else launch_few_down<NI - 1>(ni, grid, st, p);
    }
}

// Mean rows an expert up to which a form is taken.  The few-rows form reads an expert's rows once for every strip of 16
// features, the middle one once for every 128 columns but holds 64 rows in a tile; from about one of those tiles on the larger
// tiles of gemm_experts_kernel, whose waves without rows only load, need fewer loads a product and no quantiser in between.
// Whole calls, few / middle, us: 128 experts of 2048 x 768, top 8: 8 rows an expert 136 / 146, 16: 159 / 139; 32 of 3584 x 1536, top 4:
// 8: 128 / 130, 24: 175 / 116; 64 of 1024 x 512, top 6: 12: 38.7 / 37.5, 24: 49 / 44.  Middle / many: 128 of 2048 x 768: 30: 146.9 / 145.7,
// 44: 156 / 145, 48: 163 / 147, 80: 224 / 165; 64 of 2048 x 1024: 40: 101.1 / 102.3, 50: 115 / 104; 64 of 1024 x 512: 34: 45.4 / 45.6, 40: 46.7 / 45.8, 50: 57 / 47.
// The large tiles are one a CU, in rounds: where the last ones leave many CUs idle, the small ones, two a CU, stay ahead up to where
// experts come to have a second tile of 64 rows (many_idles): 32 of 3584 x 1536: 45: 121.6 / 129.7, 50: 133.2 / 133.0, 55: 146 / 137; 32 of 3584 x 1280: 46: 118.6 / 124.2,
// 50: 114.6 / 121.4, 52: 124.9 / 124.5; 32 of 2560 x 1280: 46: 94.9 / 100.1, 50: 97.1 / 100.3; 48 of 3584 x 1408: 46: 177 / 182; 24 of 3584 x 1536: 46: 111 / 120.
// Streams / middle: 128 experts of 2048 x 768: 11 rows 132.1 / 134.0, 13: 143.1 / 137.1; 32 of 3584 x 1536: 11: 105.3 / 118.5, 13: 112.3 / 116.4; 64 of 1024 x 512: 12: 36.9 / 38.9, 16: 41.9 /
// 39.4; 64 of 2048 x 1024: 12: 90.8 / 89.9.
// Where the middle form's down is down_stream_kernel and the weights are more than the memory-side cache holds, the line is at 10 rows again, between crossings that lie from 8 to beyond 12: what streams lose are
// experts with a second tile of 16 rows, which read their weights again, and how many those are, or leave CUs a second share, is not in the mean.  Weights that no cache holds, streams / middle: 128 of 2048 x 768: 6: 112.9 / 116.3,
// 8: 122.9 / 118.1, 9: 122.1 / 119.9, 10: 127.2 / 121.6, 12: 130.9 / 122.7, but 100 of them: 10: 98.4 / 105.0, 12: 105.6 / 108.2; 128 of 3584 x 640: 8: 166.8 / 167.4, 9: 173.7 / 171.5, 10: 178.0 / 172.1, 12: 191.8 / 175.2;
// 64 of 3584 x 1024: 7: 132.8 / 133.0, 8: 133.9 / 129.0, 10: 137.1 / 130.6; 32 of 3584 x 1536: 10: 104.3 / 108.4, 11: 104.0 / 108.4, 12: 117.4 / 109.2; 64 of 2048 x 1024: 9: 80.0 / 83.2, 10: 82.6 / 83.3, 11: 86.9 / 84.2;
// 128 of 1280 x 1280: 9: 127.5 / 128.5, 10: 130.1 / 129.4, 12: 138.9 / 130.9; 96 of 2560 x 896: 9: 128.6 / 129.9, 10: 132.1 / 130.6, 12: 148.1 / 134.9.  At the line it is up to 5 % either way.  Weights that the cache holds,
// 64 of 1024 x 512: 12: 37.7 / 38.6.
// Where gemm_experts_kernel does not take both products, against the other grouped GEMMs: 128 of 2048 x 768: 96: 233 / 246, 128: 266 / 256.
constexpr int64_t kFewRowsPerExpert = 10, kStreamRowsPerExpert = 12, kMiddleRowsPerExpert = 44, kMiddleRowsManyIdle = 50, kMiddleRowsElsewhere = 112;
// Many rows: up to here an expert has a second tile of 128 rows seldom enough for streaming loads of the weights to pay, if they are
// more than the memory-side cache holds (those that it holds it keeps from call to call, if loads are cacheable).  Cacheable and
// streaming, us: 128 experts of 2048 x 768 (604 MB) 48 rows an expert 167 / 161, 69: 179 / 172, 94: 185 / 180, 156: 239 / 288; 64 of 2048 x 1024 (403 MB)
// 100: 131 / 128; 64 of 2048 x 640 (252 MB) 94: 107 / 107; 64 of 1024 x 512 (101 MB) 56: 56 / 59, 112: 73 / 76.
constexpr int64_t kTileOnceRowsPerExpert = 100, kMemorySideCache = (int64_t)256 << 20;
// Up to here the weights of the middle form are loaded as a stream: an expert seldom has a second tile of 64 rows, which reads
// them again.  128 experts of 2048 x 768, rows an expert, the whole call cacheable and streaming, us: 12.5 148.8 / 137.9, 25
// 155.6 / 146.5, 49 168.4 / 163.0, 62 194.9 / 203.8, 88 232.6 / 274.3; 32 experts of 3584 x 1536: 32 134.4 / 123.4, 75
// 190.2 / 214.2.
constexpr int64_t kOnceRowsPerExpert = 52;

// Whether the last rounds of gemm_experts_kernel's tiles leave enough CUs idle for the middle form to be ahead beyond kMiddleRowsPerExpert.
// An expert is one row of tiles of 256 columns; a product of less than one round takes a tile's time however many CUs it leaves, and weights that the
// memory-side cache keeps leave nothing to wait for (32 of 2304 x 1152: 46: 83.2 / 82.6).  What the middle form loses instead grows with
// the rows: middle / many at 46 rows an expert by idle K steps a CU: 32 of 3584 x 1024 (2.0) 92.1 / 91.2, 40 of 3072 x 1280 (11.8) 126.3 / 125.8, 32 of 3584 x 1536
// (17.0) 121.6 / 130.0, 32 of 2304 x 1536 (19.5) 97.0 / 100.4, 64 of 2816 x 1152 (18.8) 159 / 157, 64 of 2304 x 1152 (20.3) 136.7 / 136.0, 64 of 3584 x 1152 (25.5) 188 / 190.
// With more columns of h than of x it is behind (32 of 2304 x 2816: 48: 153 / 148).
static bool many_idles(int64_t pairs, int64_t experts, int64_t hidden, int64_t inter) {
    const int64_t cus = cu_count();
    auto idle = [&](int64_t tiles, int64_t k) { return tiles > cus ? ((tiles + cus - 1) / cus * cus - tiles) * (k / 128) : 0; };
    const int64_t steps = idle(experts * (inter / 128), hidden) + idle(experts * ((hidden + 255) / 256), inter);
    return inter <= hidden && experts * 3 * hidden * inter > kMemorySideCache && steps * 112 >= pairs * cus;
}

// few_stream_kernel in place of the kernels of a strip a workgroup: no more tiles of 16 rows than workgroups, so that a share lies in two; some 640 strips of gate_up and more, of
// which a wave each has enough of the weights in flight; and weights of 32 MiB and more, where strips are short of 64 from a third row an expert on, of 72 and (a short
// K of gate_up) 80 with fewer rows: with less the tables and a strip's ends are what takes the time.  Beyond kFewRowsPerExpert what they stand beside is the middle form, which they are ahead of nearly everywhere (32 of 1024 x 1024, 12 rows, 39.2 / 37.7).  Whole calls on weights that no cache holds, us, strips / streams:
// 1 token of 64 experts of 3584 x 512, top 8 (512 strips, 42 MiB) 24.0 / 27.1, 2 of 8 of 3584 x 1024, top 2 (512, 42) 24.1 / 25.4, 1 of 60 of 2048 x 1408, top 4 (704, 33) 24.9 / 23.5, 1 of 32 of 3584 x 1536,
// top 4 (768, 63) 31.0 / 28.0; 2 of 128 of 1280 x 1280, top 4 (38 MiB) 26.1 / 24.9; 32 of 1024 x 512, top 4: 8 (48 MiB, a row an expert) 21.2 / 22.8, 32: 24.1 / 25.6, 96 (12 rows; middle) 30.1 / 29.3; 16 of 2048 x
// 512, top 4 (48): 8: 23.2 / 24.7, 48 (12 rows) 32.0 / 27.6; 32 of 1024 x 768, top 8 (72): 4: 25.4 / 26.9, 16: 30.3 / 29.7, 32: 32.4 / 30.8; 32 of 1152 x 640, top 4 (68): 32: 32.2 / 30.6; 2 of 128 of 3328 x 768, top 5 (73) 32.0 / 31.0; 5 of 64 of 1024 x 640, top 8 (75) 28.9 / 29.4; 64 of 1024 x 512, top 6: 8 (72) 26.4 / 27.3, 21 (96)
// 32.6 / 31.7; 128 of 2048 x 768, top 8: 1 (36) 24.6 / 25.1, 4: 42.4 / 41.0, 16: 90.6 / 81.0, 64: 126.7 / 115.6, 150: 145 / 129; 32 of 3584 x 1536, top 4: 8: 89.2 / 74.7, 60: 129 / 102.
static bool few_streams(int64_t pairs, int64_t slots, int64_t experts, int64_t hidden, int64_t inter) {
    const int64_t least = pairs > kFewRowsPerExpert * experts || (inter >= 1024 && hidden > 1024) ? 32 : pairs > 2 * experts ? 64 : hidden >= 1280 ? 72 : 80;
    return experts <= kStreamMostExperts && slots + pairs / 16 <= cu_count() && slots * (inter / 8) >= 640 && slots * 3 * hidden * inter >= least << 20;
}

enum class Form { kFew, kMiddle, kMany };
struct ExpertsPlan {
    Form form;
    int64_t rows;   // rows of the expert-grouped layout (their bound)
    int64_t slots;  // experts that can have a row
    bool gathers;   // many rows: the gate_up product reads its rows from the quantised tokens
    bool streams;   // few rows: few_stream_kernel
    int down_rows;  // middle: rows of a tile of down_stream_kernel, 0: the ring kernel
    size_t row_tokens, row_experts, row_map, weights, m_sizes, m_offsets, route, xq, xs, h, hq, hs, out, bytes;
};

static ExpertsPlan experts_plan(int64_t tokens, int topk, int experts, int64_t hidden, int64_t inter) {
    ExpertsPlan p{};
    const int64_t pairs = tokens * topk;
    p.gathers = experts_gate_up_takes(tokens, hidden, inter);
    const int64_t middle = !p.gathers || !experts_down_takes(hidden, inter) ? kMiddleRowsElsewhere : many_idles(pairs, experts, hidden, inter) ? kMiddleRowsManyIdle : kMiddleRowsPerExpert;
    p.slots = pairs < experts ? pairs : experts;
    p.streams = few_streams(pairs, p.slots, experts, hidden, inter);
    p.down_rows = down_stream_rows(pairs, p.slots, experts, hidden, inter);
    const bool behind = p.down_rows && ring_grouped_takes(hidden) && ring_grouped_takes(inter) && (int64_t)experts * 3 * hidden * inter > kMemorySideCache;
    const int64_t few = p.streams && !behind ? kStreamRowsPerExpert : kFewRowsPerExpert;
    if (pairs <= few * experts && hidden <= kFewMaxHidden && inter <= kFewMaxInter) p.form = Form::kFew;
    else if (pairs <= middle * experts && ring_grouped_takes(hidden) && ring_grouped_takes(inter) && tokens * hidden < (int64_t)1 << 31) p.form = Form::kMiddle;
    else p.form = Form::kMany;
    const bool many = p.form == Form::kMany;
    p.rows = many ? (pairs + p.slots * 127) / 128 * 128 : pairs;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += (bytes + 255) & ~(size_t)255;
        return here;
    };
    p.row_tokens = take((size_t)p.rows * 4);
    p.row_experts = take(many ? (size_t)p.rows * 4 : 0);
    p.row_map = take((size_t)pairs * 4);
    p.weights = take((size_t)pairs * 2);
    p.m_sizes = take((size_t)experts * 4);
    p.m_offsets = take((size_t)experts * 4);
    p.route = take(cfp8_route_tokens_workspace_bytes(tokens, topk, experts));
    p.gathers = p.gathers && many;
    const size_t xrows = (size_t)(many && !p.gathers ? p.rows : tokens);
    p.xq = take(xrows * (size_t)hidden);
    p.xs = take(xrows * (size_t)(hidden / 128) * 4);
    p.h = take(many ? 0 : (size_t)p.rows * (size_t)inter * 2);
    p.hq = take(p.form == Form::kFew ? 0 : (size_t)p.rows * (size_t)inter);
    p.hs = take(p.form == Form::kFew ? 0 : (size_t)p.rows * (size_t)(inter / 128) * 4);
    p.out = take((size_t)p.rows * (size_t)hidden * 2);
    p.bytes = at;
    return p;
}

}  // namespace cfp8

extern "C" size_t cfp8_moe_experts_workspace_bytes(int64_t tokens, int topk, int experts, int64_t hidden, int64_t inter) {
    if (tokens <= 0 || topk <= 0 || experts <= 0 || hidden <= 0 || inter <= 0) return 0;
    return cfp8::experts_plan(tokens, topk, experts, hidden, inter).bytes;
}

extern "C" int cfp8_moe_experts_form(int64_t tokens, int topk, int experts, int64_t hidden, int64_t inter, char* buf, size_t buf_bytes) {
    using namespace cfp8;
    if (!buf || buf_bytes == 0) return set_error(CFP8_EINVAL, "moe_experts_form: no buffer");
    buf[0] = 0;
    if (tokens <= 0 || topk <= 0 || topk > 64 || experts <= 0 || hidden <= 0 || inter <= 0 || hidden % 128 || inter % 128 || tokens > 0x7FFFFFFFll / 64)
        return set_error(CFP8_EINVAL, "moe_experts_form: bad shape");
    const ExpertsPlan p = experts_plan(tokens, topk, experts, hidden, inter);
    if (p.form == Form::kFew) snprintf(buf, buf_bytes, "few %s", p.streams ? "streams" : "strips");
    else if (p.form == Form::kMany) snprintf(buf, buf_bytes, "many gate_up=%s down=%s", p.gathers ? "experts" : "grouped", experts_down_takes(hidden, inter) ? "experts" : "grouped");
    else if (p.down_rows) snprintf(buf, buf_bytes, "middle down=streams,%d", p.down_rows);
    else snprintf(buf, buf_bytes, "middle down=ring");
    return CFP8_OK;
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
    // the tokens quantised as they lie, for the products that pick their rows themselves
    const bool as_they_lie = p.form != Form::kMany || p.gathers;
    if (as_they_lie && tokens * (hidden / 128) > kMaxGroups) return set_error(CFP8_EINVAL, "moe_experts: too many groups for one launch");
    const GroupRows xq = group_rows(x, tokens, hidden, ld_x, ws + p.xq, hidden, f32(p.xs));
    if (int rc = route_and_quantise(indices, index_bytes, token_mask, tokens, topk, experts, p.form == Form::kMany ? 128 : 1, CFP8_ROUTE_END_NOT_PADDING, p.rows,
                                    i32(p.row_tokens), p.form == Form::kMany ? i32(p.row_experts) : nullptr, i32(p.row_map), nullptr, weights, weights_dtype,
                                    ws + p.weights, i32(p.m_sizes), i32(p.m_offsets), ws + p.route, cfp8_route_tokens_workspace_bytes(tokens, topk, experts),
                                    as_they_lie ? &xq : nullptr, st))
        return rc;
    if (p.form == Form::kMiddle) {
        const int64_t row_tiles = p.slots + p.rows / kRingGroupRows;
        const bool once = p.rows <= kOnceRowsPerExpert * experts;
        RingArgs r{};
        r.a = ws + p.xq; r.w = static_cast<const uint8_t*>(gate_up); r.sa = f32(p.xs); r.sb = gate_up_scales; r.out = ws + p.h;
        r.ld_a = r.ld_w = hidden; r.ld_out = inter;
        r.row_tokens = i32(p.row_tokens); r.sizes = i32(p.m_sizes); r.ends = i32(p.m_offsets);
        r.experts = experts;
        r.M = (int)tokens; r.N = (int)(2 * inter); r.K = (int)hidden;
        if (int rc = launch_ring_grouped(kRingGateUp, r, row_tiles, once, st)) return rc;
        if (int rc = cfp8_quant_group128(ws + p.h, p.rows, inter, inter, ws + p.hq, inter, f32(p.hs), CFP8_GROUP_MODE_DIV, stream)) return rc;
        if (const int tile = p.down_rows) {
            DownArgs d{};
            d.hq = ws + p.hq; d.hs = f32(p.hs); d.w = static_cast<const uint8_t*>(down); d.ws = down_scales;
            d.sizes = i32(p.m_sizes); d.out = reinterpret_cast<uint16_t*>(ws + p.out);
            d.experts = experts; d.hidden = (int)hidden; d.inter = (int)inter;
            if (int rc = tile == 64 ? launch_down_stream<4>(d, st) : tile == 48 ? launch_down_stream<3>(d, st) : launch_down_stream<2>(d, st)) return rc;
        } else {
            r.a = ws + p.hq; r.w = static_cast<const uint8_t*>(down); r.sa = f32(p.hs); r.sb = down_scales; r.out = ws + p.out;
            r.ld_a = r.ld_w = inter; r.ld_out = hidden;
            r.M = (int)p.rows; r.N = (int)hidden; r.K = (int)inter;
            if (int rc = launch_ring_grouped(kRingDown, r, row_tiles, once, st)) return rc;
        }
    } else if (p.form == Form::kFew) {
        FewArgs f{};
        f.xq = ws + p.xq;
        f.xs = f32(p.xs);
        f.w = static_cast<const uint8_t*>(gate_up);
        f.ws = gate_up_scales;
        f.row_tokens = i32(p.row_tokens);
        f.sizes = i32(p.m_sizes);
        f.ends = i32(p.m_offsets);
        f.h = reinterpret_cast<uint16_t*>(ws + p.h);
        f.out = reinterpret_cast<uint16_t*>(ws + p.out);
        f.experts = experts;
        f.hidden = (int)hidden;
        f.inter = (int)inter;
        if (p.streams) {
            f.tokens = (int)tokens;
            if (int rc = launch_few_stream<false>(f, st)) return rc;
            f.w = static_cast<const uint8_t*>(down);
            f.ws = down_scales;
            if (int rc = launch_few_stream<true>(f, st)) return rc;
        } else {
            launch_few_gate_up<(int)(kFewMaxHidden / 512)>((int)((hidden / 128 + 3) / 4), dim3((unsigned)(inter / 16), (unsigned)p.slots), st, f);
            f.w = static_cast<const uint8_t*>(down);
            f.ws = down_scales;
            launch_few_down<(int)(kFewMaxInter / 128)>((int)(inter / 128), dim3((unsigned)(hidden / 128), (unsigned)p.slots), st, f);
            if (int rc = check_launch("moe_experts")) return rc;
        }
    } else {
        // (p.rows is a bound: 639 tiles of rows for 8192 tokens, top 8 of 128 experts, of which some 566 hold rows)
        const int32_t* const rows_end = i32(p.m_offsets) + experts - 1;
        const bool once = tokens * topk <= kTileOnceRowsPerExpert * experts && (int64_t)experts * 3 * hidden * inter > kMemorySideCache;
        if (p.gathers) {
            ExpertsArgs g{};
            g.x = ws + p.xq; g.xs = f32(p.xs); g.w = static_cast<const uint8_t*>(gate_up); g.ws = gate_up_scales;
            g.row_tokens = i32(p.row_tokens); g.row_experts = i32(p.row_experts); g.rows_end = rows_end;
            g.h = ws + p.hq; g.hs = f32(p.hs);
            g.tokens = (int)tokens; g.N = (int)(2 * inter); g.K = (int)hidden;
            g.whole_tiles = !experts_down_takes(hidden, inter);
            if (int rc = launch_experts_gate_up(g, p.rows, once, st)) return rc;
        } else {
            if (int rc = cfp8_scatter_quant_group128(x, ld_x, tokens, hidden, i32(p.row_map), topk, i32(p.row_tokens), p.rows, ws + p.xq, hidden, f32(p.xs), stream))
                return rc;
            if (int rc = cfp8_gemm_grouped_swiglu_quant(ws + p.xq, hidden, f32(p.xs), gate_up, gate_up_scales, i32(p.row_experts), ws + p.hq, inter,
                                                        f32(p.hs), p.rows, inter, hidden, experts, stream))
                return rc;
        }
        if (experts_down_takes(hidden, inter)) {
            ExpertsArgs d{};
            d.x = ws + p.hq; d.xs = f32(p.hs); d.w = static_cast<const uint8_t*>(down); d.ws = down_scales;
            d.row_tokens = i32(p.row_tokens); d.row_experts = i32(p.row_experts); d.rows_end = rows_end; d.out = reinterpret_cast<uint16_t*>(ws + p.out);
            d.N = (int)hidden; d.K = (int)inter;
            if (int rc = launch_experts_down(d, p.rows, once, st)) return rc;
        } else {
            if (int rc = cfp8_gemm_grouped_block128(ws + p.hq, inter, f32(p.hs), down, down_scales, i32(p.row_experts), ws + p.out, hidden, CFP8_OUT_BF16,
                                                    p.rows, hidden, inter, experts, stream))
                return rc;
        }
    }
    return cfp8_combine_rows(ws + p.out, hidden, p.rows, i32(p.row_map), ws + p.weights, CFP8_IN_BF16, tokens, topk, hidden,
                             CFP8_COMBINE_BF16_STEPS, y, ld_y, stream);
}
