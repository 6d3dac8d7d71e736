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
//               kRingGateUp reads them from the quantised tokens and ends in SwiGLU, kRingDown), two workgroups a CU.  The
//               hidden activation is quantised in between, since a 1x128 group of it is spread over two workgroups.
//   few rows    A decode batch: reading the weights of the experts that have a row is all the time there is, and tiles of
//               64 rows would hold one or two.  A workgroup takes a strip of ONE expert's weight rows, requests all of its
//               K into registers before anything else, and then walks the expert's rows in tiles of 16
//               (few_gate_up_kernel, few_down_kernel).
#include "gemm_internal.h"
#include "moe_route.h"
#include "gemm_ring.h"

namespace cfp8 {

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
    int experts, hidden, inter;
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

// The few-rows form holds a strip's whole K in registers: up to 8 K steps a wave of four (gate_up, 128 registers of weights and 64 of
// tokens), 12 a wave (down, 96 registers, and two tiles of 16 rows of 1536 bytes in LDS).
constexpr int64_t kFewMaxHidden = 4096, kFewMaxInter = 1536;
// Mean rows an expert up to which a form is taken.  The few-rows form reads an expert's rows once for every strip of 16
// features, the middle one once for every 128 columns but holds 64 rows in a tile; from about one of those tiles on the larger
// tiles of gemm_experts_kernel, whose waves without rows only load, need fewer loads a product and no quantiser in between.
// Whole calls, few / middle, us: 128 experts of 2048 x 768, top 8: 8 rows an expert 136 / 146, 16: 159 / 139; 32 of 3584 x 1536, top 4:
// 8: 128 / 130, 24: 175 / 116; 64 of 1024 x 512, top 6: 12: 38.7 / 37.5, 24: 49 / 44.  Middle / many: 128 of 2048 x 768: 30: 146.9 / 145.7,
// 44: 156 / 145, 48: 163 / 147, 80: 224 / 165; 64 of 2048 x 1024: 40: 101.1 / 102.3, 50: 115 / 104; 64 of 1024 x 512: 34: 45.4 / 45.6, 40: 46.7 / 45.8, 50: 57 / 47.
// The large tiles are one a CU, in rounds: where the last ones leave many CUs idle, the small ones, two a CU, stay ahead up to where
// experts come to have a second tile of 64 rows (many_idles): 32 of 3584 x 1536: 45: 121.6 / 129.7, 50: 133.2 / 133.0, 55: 146 / 137; 32 of 3584 x 1280: 46: 118.6 / 124.2,
// 50: 114.6 / 121.4, 52: 124.9 / 124.5; 32 of 2560 x 1280: 46: 94.9 / 100.1, 50: 97.1 / 100.3; 48 of 3584 x 1408: 46: 177 / 182; 24 of 3584 x 1536: 46: 111 / 120.
// Where gemm_experts_kernel does not take both products, against the other grouped GEMMs: 128 of 2048 x 768: 96: 233 / 246, 128: 266 / 256.
constexpr int64_t kFewRowsPerExpert = 10, kMiddleRowsPerExpert = 44, kMiddleRowsManyIdle = 50, kMiddleRowsElsewhere = 112;
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

enum class Form { kFew, kMiddle, kMany };
struct ExpertsPlan {
    Form form;
    int64_t rows;   // rows of the expert-grouped layout (their bound)
    int64_t slots;  // experts that can have a row
    bool gathers;   // many rows: the gate_up product reads its rows from the quantised tokens
    size_t row_tokens, row_experts, row_map, weights, m_sizes, m_offsets, route, xq, xs, h, hq, hs, out, bytes;
};

static ExpertsPlan experts_plan(int64_t tokens, int topk, int experts, int64_t hidden, int64_t inter) {
    ExpertsPlan p{};
    const int64_t pairs = tokens * topk;
    p.gathers = experts_gate_up_takes(tokens, hidden, inter);
    const int64_t middle = !p.gathers || !experts_down_takes(hidden, inter) ? kMiddleRowsElsewhere : many_idles(pairs, experts, hidden, inter) ? kMiddleRowsManyIdle : kMiddleRowsPerExpert;
    if (pairs <= kFewRowsPerExpert * experts && hidden <= kFewMaxHidden && inter <= kFewMaxInter) p.form = Form::kFew;
    else if (pairs <= middle * experts && ring_grouped_takes(hidden) && ring_grouped_takes(inter) && tokens * hidden < (int64_t)1 << 31) p.form = Form::kMiddle;
    else p.form = Form::kMany;
    const bool many = p.form == Form::kMany;
    p.slots = pairs < experts ? pairs : experts;
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
        r.a = ws + p.hq; r.w = static_cast<const uint8_t*>(down); r.sa = f32(p.hs); r.sb = down_scales; r.out = ws + p.out;
        r.ld_a = r.ld_w = inter; r.ld_out = hidden;
        r.M = (int)p.rows; r.N = (int)hidden; r.K = (int)inter;
        if (int rc = launch_ring_grouped(kRingDown, r, row_tiles, once, st)) return rc;
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
        launch_few_gate_up<(int)(kFewMaxHidden / 512)>((int)((hidden / 128 + 3) / 4), dim3((unsigned)(inter / 16), (unsigned)p.slots), st, f);
        f.w = static_cast<const uint8_t*>(down);
        f.ws = down_scales;
        launch_few_down<(int)(kFewMaxInter / 128)>((int)(inter / 128), dim3((unsigned)(hidden / 128), (unsigned)p.slots), st, f);
        if (int rc = check_launch("moe_experts")) return rc;
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
