// The ring kernel's form for few rows (included by gemm_ring.hip): all rows in one tile, every wave a strip of 16 weight rows of its own.
// Rowwise up to 256 rows, MXFP4 255, block-scaled 128.
//
// Bound by the weights' way in, and behind it by the activations, which every workgroup loads and every wave reads from LDS.  A wave reads its strip, 8 rows x 128 bytes a
// load, into a ring of its own that no barrier guards; the workgroup shares the activations, a chunk of one or two K steps of all
// rows, and has one barrier a chunk.  So a workgroup can have any number of strips, and the weight is dealt to the CUs evenly, one
// workgroup each: 2368 strips as 237 workgroups of ten, where tiles of 64 x 64 are 592 on 512 places and load the activations 592 times.
// Three or four K steps a wave are enough in flight (as a stream alone, 132 MB on 144 workgroups of eight waves, 4, 6 and 9 steps: 23.7, 23.7 and 24.0 us);
// a fragment's own address pattern straight into registers, 16 rows at a time, stops at 5 TB/s where this one reaches 6.2.
// Products, us, tiles of the ring kernel / this form, weights cold: 5 x 37888 x 3584 26.6 / 22.6, 33: 28.7 / 24.3, 64: 33.1 / 25.9, 128: 43.9 / 31.8,
// 200: 56.5 / 43.3, 256: 65.0 / 48.3; 33 x 25344 x 2560 15.2 / 14.2; block-scaled 24 x 18432 x 7168 30.3 / 23.5, 64: 35.2 / 29.5, 100: 47.0 / 40.0.
// MXFP4: 5 x 37888 x 3584 26.2 / 15.7, 33: 30.9 / 18.4, 128: 44.8 / 28.5, 200: 46.3 / 39.5; 33 x 18944 x 3584 17.3 / 12.3.
// MXFP4, 200 rows: a step takes 1.4 us.  The 39 products on the fullest SIMD are 0.6 of it; ten waves that each read 26 KiB of activations and 1 of weights from LDS are 0.9 at 128 bytes a cycle.
// Two or three strips a wave, whose fragments are read half or a third as often, take 47 and 76 us with their four to six waves, chunks of two steps and other depths no less.
// Sums and scales are taken in the order of K as in the tiles of the ring kernel, and have their bits.
#pragma once

#include "gemm_internal.h"
#include "gemm_ring.h"

namespace cfp8 {

// TM: tiles of 16 rows.  A chunk of activations is CH K steps, XB chunks are in LDS.  A wave has D stages of its strips in LDS, a K step of them each, MXFP4 two: 128 bytes of a row.
// WIDTH: workgroups of 3 waves (up to 32 rows), of 4 to 7 (rowwise up to 80 rows, the others 128), of 8 to 12.
// The waves share out a chunk's loads of 1 KiB; where these do not share out evenly some load nothing to nowhere, so that all count the same.
constexpr int few_threads(int width) { return (width == 0 ? 3 : width == 1 ? 7 : 12) * 64; }
constexpr int few_steps(int tm) { return tm <= 8 ? 2 : 1; }
constexpr int few_chunks(int tm) { return tm <= 4 || tm > 8 ? 3 : 2; }
constexpr int few_depth(int mode, int tm) { return mode == kRingMx ? (tm <= 2 ? 3 : 2) : tm <= 2 || (tm > 8 && tm <= 13) ? 4 : 3; }
constexpr int few_stage(int mode) { return 2048 + (mode == kRingMx ? 256 : 0); }
// Whether 16-byte chunk `chunk` of a row's 128 in a stage of MXFP4 weights that begins with K step kt holds codes below K (or below a slice's end): a
// stage is two steps, and the codes of an odd last one end in its middle.  Behind them lies the next row or, where rows have a pitch, what may not be mapped.
__host__ __device__ constexpr bool few_codes_inside(int kt, uint32_t chunk, uint32_t K) { return ((uint32_t)kt << 7) + chunk * 32 < K; }
constexpr bool few_codes_stay_in_their_rows() {
    for (uint32_t K = 32; K <= 4096; K += 32) {
        uint32_t loaded = 0;
        for (int kt = 0; kt < (int)((K + 127) / 128) + 4; kt += 2)
            for (uint32_t c = 0; c < 8; ++c)
                if (few_codes_inside(kt, c, K)) {
                    if (((uint32_t)kt << 6) + c * 16 + 16 > K / 2) return false;
                    loaded += 16;
                }
        if (loaded != K / 2) return false;
    }
    return true;
}
static_assert(few_codes_stay_in_their_rows(), "stages of MXFP4 weights read all of a row's codes and nothing behind them");
template <int MODE, int TM, int WIDTH>
struct FewShape {
    static constexpr int CH = few_steps(TM), D = few_depth(MODE, TM), STAGE = few_stage(MODE);
    static constexpr int WK = MODE == kRingMx ? 2 : 1, WL = MODE == kRingMx ? 3 : 2;  // K steps and loads of a stage of weights
    static constexpr int XSTEP = TM * 2048, XS = CH * XSTEP, WS = D * STAGE;
    static constexpr int XB = few_chunks(TM);
    static constexpr int LOADS = TM * 2 * CH, LEAST = WIDTH == 0 ? 3 : WIDTH == 1 ? 4 : 8;
    static constexpr int XL = (LOADS + LEAST - 1) / LEAST;
    static constexpr int NOWHERE = XB * XS, WB = NOWHERE + 1024;
    static_assert(CH <= D * WK && (CH % WK == 0 || CH == 1), "a step's weights are requested before its chunk begins");
};

template <int MODE, int TM, int WIDTH>
__global__ __launch_bounds__(few_threads(WIDTH)) void gemm_ring_few_kernel(const RingArgs p, const int f32) {
    using Sh = FewShape<MODE, TM, WIDTH>;
    constexpr int CH = Sh::CH, XB = Sh::XB, D = Sh::D, XL = Sh::XL, WK = Sh::WK, STAGE = Sh::STAGE;
    constexpr bool MX = MODE == kRingMx;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    typedef __attribute__((address_space(3))) void lds_void;
    const int t = threadIdx.x, lane = t & 63, NW = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lrow = lane & 15, quarter = lane >> 4;
    const int slice = (int)blockIdx.x / p.tiles_n;
    const int pid = (int)blockIdx.x - slice * p.tiles_n;
    const int xcd = pid & 7, local = pid >> 3, base = p.tiles_n >> 3, rem = p.tiles_n & 7;
    const int n0 = (xcd * base + (xcd < rem ? xcd : rem) + local) * NW * 16;
    const int KT = (p.K + 127) >> 7, tail = p.K & 127;
    const int kbeg = slice * p.slice_steps;
    const int kend = kbeg + p.slice_steps < KT ? kbeg + p.slice_steps : KT;
    const int steps = kend - kbeg, chunks = (steps + CH - 1) / CH;

    constexpr uint32_t kMost = 0xEFFFFFFFu;
    auto bytes = [&](int64_t rows, int64_t ld) -> uint32_t {
        const int64_t b = rows > 0 ? rows * ld : 0;
        return b < (int64_t)kMost ? (uint32_t)b : kMost;
    };
    const int nw0 = n0 + wave * 16;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.a), 0, (int)bytes(p.M, p.ld_a), 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w) + (uint64_t)nw0 * (uint64_t)p.ld_w, 0, (int)bytes((int64_t)p.N - nw0, p.ld_w), 0x00020000);
    // a load of 8 rows x 128 bytes: row lane >> 3, whose 16-byte chunk c lies at position c ^ f(row) (gemm_ring.hip; the half says rows 8 .. 15 of 16)
    constexpr int F1 = MX ? 1 : 0;
    auto chunk_of = [&](int half) { return (uint32_t)((lane & 7) ^ ((((lane >> 4) & 1) << F1) | (half << 2))); };
    uint32_t vw[2], vw_tail[2], vx[XL], vx_tail[XL];  // (MXFP4: vw_tail is the load's chunk)
    int xstep[XL], xdst[XL], xbuf[XL];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t c = chunk_of(h);
        vw[h] = (uint32_t)((lane >> 3) + 8 * h) * (uint32_t)p.ld_w + c * 16;
        vw_tail[h] = MX ? c : tail && c * 16 >= (uint32_t)tail ? kOutside : vw[h];
    }
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int l = wave + NW * i, j = l / (2 * TM), g = l - j * 2 * TM;
        const bool real = l < Sh::LOADS;
        const uint32_t c = chunk_of(g & 1);
        xstep[i] = j;
        xdst[i] = real ? l * 1024 : Sh::NOWHERE;
        xbuf[i] = real ? Sh::XS : 0;
        vx[i] = real ? (uint32_t)((lane >> 3) + 8 * g) * (uint32_t)p.ld_a + c * 16 : kOutside;
        vx_tail[i] = tail && c * 16 >= (uint32_t)tail ? kOutside : vx[i];
    }
    auto dma_x = [&](int c, int buf) {
#pragma unroll
        for (int i = 0; i < XL; ++i) {
            const int kt = kbeg + c * CH + xstep[i];
            const uint32_t v = kt < kend ? (kt == KT - 1 ? vx_tail[i] : vx[i]) : kOutside;
            uint8_t* const to = smem + buf * xbuf[i] + xdst[i];
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void*)to, 16, v, (uint32_t)kt << 7, 0, 0);
        }
    };
    uint8_t* const own = smem + Sh::WB + wave * Sh::WS;
    const uint32_t klimit = kend < KT ? (uint32_t)kend << 7 : (uint32_t)p.K;
    const __amdgpu_buffer_rsrc_t rsc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(MX ? p.ws + (uint64_t)nw0 * (uint64_t)p.ld_ws : p.w), 0,
                                                                         MX ? (int)bytes((int64_t)p.N - nw0, p.ld_ws) : 0, 0x00020000);
    auto dma_w = [&](int kt, int st) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint32_t v;
            if (MX) v = few_codes_inside(kt, vw_tail[h], klimit) ? vw[h] : kOutside;
            else v = kt < kend ? (kt == KT - 1 ? vw_tail[h] : vw[h]) : kOutside;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_void*)(own + st * STAGE + h * 1024), 16, v, (uint32_t)kt << (MX ? 6 : 7), 0, 2);
        }
        if (MX) {
            // lanes 16 s .. 16 s + 15: the four scale bytes of step kt + s of a row; of a step that is shorter the four that end with the row
            const int ks = kt + ((lane >> 4) & 1);
            const uint32_t at = ks == KT - 1 && tail ? (uint32_t)(p.K >> 5) - 4u : (uint32_t)ks << 2;
            const uint32_t v = lane < 32 && ks < kend ? (uint32_t)lrow * (uint32_t)p.ld_ws + at : kOutside;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsc, (lds_void*)(own + st * STAGE + 2048), 4, v, 0, 0, 0);
        }
    };
    // block scaling: the slice's activation scales, [row][step], and the weight scales of the blocks that the workgroup's strips lie
    // in, requested in front of everything else
    uint8_t* const scales = smem + Sh::WB + NW * Sh::WS;
    const float* const sa_lds = reinterpret_cast<const float*>(scales);
    const int pitch = steps | 1, sa_words = (p.M * pitch + 63) & ~63, sb_words = (steps + 63) & ~63;
    const float* const sb_lds = sa_lds + sa_words + ((nw0 >> 7) - (n0 >> 7)) * sb_words;
    if (MODE == kRingBlock) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.sa), 0, p.M * KT * 4, 0x00020000);
        for (int e0 = wave * 64; e0 < p.M * pitch; e0 += NW * 64) {
            const int e = e0 + lane, r = e / pitch, c = e - r * pitch;
            uint8_t* const to = scales + e0 * 4;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)to, 4, c < steps ? (uint32_t)(r * KT + kbeg + c) * 4u : kOutside, 0, 0, 0);
        }
        const int end = n0 + NW * 16 < p.N ? n0 + NW * 16 : p.N, blocks = ((end - 1) >> 7) - (n0 >> 7) + 1;
        const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.sb) + (int64_t)(n0 >> 7) * p.sb_stride_n, 0,
                                                                            (int)((blocks - 1) * p.sb_stride_n + (KT - 1) * p.sb_stride_k + 1) * 4, 0x00020000);
        for (int e0 = wave * 64; e0 < blocks * sb_words; e0 += NW * 64) {
            const int b = e0 / sb_words, c = e0 - b * sb_words + lane;
            uint8_t* const to = scales + (sa_words + e0) * 4;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void*)to, 4, c < steps ? (uint32_t)(b * p.sb_stride_n + (kbeg + c) * p.sb_stride_k) * 4u : kOutside, 0, 0, 0);
        }
    }
#pragma unroll
    for (int c = 0; c < XB - 1; ++c) dma_x(c, c);
#pragma unroll
    for (int d = 0; d < D; ++d) dma_w(kbeg + d * WK, d);

    // fragments: the lane's two chunks of a row, MXFP4 weights have one
    const int fr = (((lrow >> 1) & 1) << F1) | (((lrow >> 3) & 1) << 2);
    const int fo = lrow * 128 + (((MX ? quarter : 2 * quarter) ^ fr) << 4), other = MX ? 64 : 16;
    auto frag = [&](const uint8_t* at) {
        const i32x4 lo = *reinterpret_cast<const i32x4*>(at + fo);
        const i32x4 hi = *reinterpret_cast<const i32x4*>(at + (fo ^ other));
        return i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    auto wfrag = [&](const uint8_t* at, int s) {
        if (!MX) return frag(at);
        const i32x4 v = *reinterpret_cast<const i32x4*>(at + (fo ^ (s * 64)));
        return i32x8{v[0], v[1], v[2], v[3], 0, 0, 0, 0};
    };
    f32x4 acc[TM];
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    int ws = 0;
    auto chunk = [&](int c, int buf, auto first_c, auto odd_c) {
        constexpr int odd = decltype(odd_c)::value;  // the first step's place in its stage of weights
        // This chunk's activations have landed when at most what was requested behind them is outstanding; every wave has read the
        // chunk before, whose place the chunk XB - 1 ahead takes.
        if constexpr (decltype(first_c)::value) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(Sh::WL * Sh::D + (Sh::XB - 2) * Sh::XL) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((Sh::XB - 2) * Sh::XL + Sh::WL * (Sh::XB - 1) * Sh::CH / Sh::WK) : "memory");
        dma_x(c + XB - 1, buf == 0 ? XB - 1 : buf - 1);
        const uint8_t* const xb = smem + buf * Sh::XS;
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const int k = c * CH + j;
            if (k < steps) {
                const int s = (odd + j) % WK;
                // its weights: behind them D - 1 stages and at least the activations just requested
                if (s == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Sh::WL * (Sh::D - 1) + Sh::XL) : "memory");
                const i32x8 w = wfrag(own + ws * STAGE, s);
                int wsc = 0;
                if (MX) {
                    u32 v = *reinterpret_cast<const u32*>(own + ws * STAGE + 2048 + s * 64 + lrow * 4);
                    if (tail && kbeg + k == KT - 1) v >>= (u32)(4 - (tail >> 5)) * 8;
                    wsc = (int)(v >> (quarter * 8));
                }
                float f[TM];
                if (MODE == kRingBlock) {
                    const float s = sb_lds[k];
#pragma unroll
                    for (int m = 0; m < TM; ++m) {
                        const int row = m * 16 + lrow;
                        f[m] = sa_lds[(row < p.M ? row : 0) * pitch + k] * s;
                    }
                }
                // (many rows: a group's fragments are read under the products of the group before, all of them at once have no registers)
                constexpr int G = TM > 8 ? 4 : TM;
                i32x8 x[2][G];
                auto read = [&](int m0) {
#pragma unroll
                    for (int m = m0; m < m0 + G && m < TM; ++m) x[m0 / G & 1][m - m0] = frag(xb + j * Sh::XSTEP + m * 2048);
                };
                read(0);
#pragma unroll
                for (int m0 = 0; m0 < TM; m0 += G) {
                    if (m0 + G < TM) read(m0 + G);
                    if (TM > G) CFP8_PHASE_END();
#pragma unroll
                    for (int m = m0; m < m0 + G && m < TM; ++m) {
                        const i32x8 xf = x[m0 / G & 1][m - m0];
                        if (MODE == kRingBlock) {
                            const f32x4 pr = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, xf, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[m][e] = __builtin_fmaf(pr[e], f[m], acc[m][e]);
                        } else if (MX) {
                            acc[m] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, xf, acc[m], 4, 0, 0, wsc, 0, 0x7F7F7F7F);
                        } else {
                            acc[m] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, xf, acc[m], 0, 0, 0, 0, 0, 0);
                        }
                        if (TM > G) asm volatile("" : "+v"(acc[m]));
                    }
                    if (TM > G) CFP8_PHASE_END();
                }
                // the last product waits for the last fragment, so that all of them have been read where the stage is given away
                asm volatile("" : "+v"(acc[TM - 1]));
                CFP8_PHASE_END();
                if (s == WK - 1) {
                    dma_w(kbeg + k + 1 + (D - 1) * WK, ws);
                    ws = ws == D - 1 ? 0 : ws + 1;
                }
            }
        }
    };
    using yes = std::integral_constant<bool, true>;
    using no = std::integral_constant<bool, false>;
    chunk(0, 0, yes{}, std::integral_constant<int, 0>{});
    int buf = 1;
    auto next = [&]() { buf = buf == XB - 1 ? 0 : buf + 1; };
    if constexpr (CH < WK) {
        // (an exit in the middle of the round would give the accumulators two sets of registers)
        int c = 1;
        for (; c + 1 < chunks; c += 2) {
            chunk(c, buf, no{}, std::integral_constant<int, 1>{});
            next();
            chunk(c + 1, buf, no{}, std::integral_constant<int, 0>{});
            next();
        }
        if (c < chunks) chunk(c, buf, no{}, std::integral_constant<int, 1>{});
    } else {
        for (int c = 1; c < chunks; ++c, next()) chunk(c, buf, no{}, std::integral_constant<int, 0>{});
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may land in LDS once the workgroup has gone

    const int n = nw0 + quarter * 4;
    if (n >= p.N) return;
    if (p.slices > 1) {
        float* const part = p.partial + (int64_t)slice * p.M * p.N + n;
#pragma unroll
        for (int j = 0; j < TM; ++j) {
            const int m = j * 16 + lrow;
            if (m < p.M) *reinterpret_cast<f32x4*>(part + (int64_t)m * p.N) = acc[j];
        }
        return;
    }
    const f32x4 sbn = MODE == kRingRow ? *reinterpret_cast<const f32x4*>(p.sb + n) : f32x4{1.f, 1.f, 1.f, 1.f};
    const uint2 bia = p.bias ? *reinterpret_cast<const uint2*>(p.bias + n) : make_uint2(kNoBias, kNoBias);
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        const int m = j * 16 + lrow;
        if (m >= p.M) continue;
        const float sam = MODE != kRingBlock ? p.sa[m] : 1.f;
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[j][e] * sam * sbn[e];
        if (f32) {
            *reinterpret_cast<f32x4*>(static_cast<float*>(p.out) + (int64_t)m * p.ld_out + n) = plus_bias<true>(v, bia.x, bia.y);
        } else {
            v = plus_bias<false>(v, bia.x, bia.y);
            *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.out) + (int64_t)m * p.ld_out + n) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
        }
    }
}

// The linear of up to four tokens on a wide weight as one launch: the same streams, and the tokens quantised by every workgroup under their first loads, a wave a
// token, into LDS (V 16-byte vectors of a token a lane: K <= 512 V).  Step k is added to the sum k mod 4 and the four sums at the end, as the four waves of
// the kernels for up to 16 rows have them, whose bits these are.  No barrier behind the tokens.
// One launch of those kernels / this one, us: rowwise 1 x 37888 x 3584 28.9 / 23.2, 4: 35.6 / 23.1, 1 x 18944 x 3584 16.2 / 13.9, 4: 20.0 / 13.2, 1 x 37888 x 8192 61.3 / 56.0; MXFP4 1 x 37888 x 3584
// 26.2 / 16.0, 4: 31.4 / 16.3, 3 x 24576 x 1024 17.0 / 6.3.
template <int MODE, int V>
__global__ __launch_bounds__(12 * 64) void linear_stream_kernel(const RingArgs p, const uint4* __restrict__ x, int64_t ldx, const int f32) {
    constexpr bool MX = MODE == kRingMx;
    constexpr int D = few_depth(MODE, 1), STAGE = few_stage(MODE), WK = MX ? 2 : 1, WL = MX ? 3 : 2;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    typedef __attribute__((address_space(3))) void lds_void;
    const int t = threadIdx.x, lane = t & 63, NW = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lrow = lane & 15, quarter = lane >> 4;
    const int KT = p.K >> 7, nvec = p.K >> 3;
    const int nw0 = ((int)blockIdx.x * NW + wave) * 16;
    uint4 v[V];
    if (wave < p.M) {
#pragma unroll
        for (int j = 0; j < V; ++j) v[j] = lane + 64 * j < nvec ? x[(int64_t)wave * ldx + lane + 64 * j] : make_uint4(0, 0, 0, 0);
    }
    auto bytes = [&](int64_t rows, int64_t ld) -> uint32_t {
        const int64_t b = rows > 0 ? rows * ld : 0;
        return b < (int64_t)0xEFFFFFFFu ? (uint32_t)b : 0xEFFFFFFFu;
    };
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w) + (uint64_t)nw0 * (uint64_t)p.ld_w, 0, (int)bytes((int64_t)p.N - nw0, p.ld_w), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(MX ? p.ws + (uint64_t)nw0 * (uint64_t)p.ld_ws : p.w), 0,
                                                                         MX ? (int)bytes((int64_t)p.N - nw0, p.ld_ws) : 0, 0x00020000);
    constexpr int F1 = MX ? 1 : 0;
    uint32_t vw[2], chunk[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        chunk[h] = (uint32_t)((lane & 7) ^ ((((lane >> 4) & 1) << F1) | (h << 2)));
        vw[h] = (uint32_t)((lane >> 3) + 8 * h) * (uint32_t)p.ld_w + chunk[h] * 16u;
    }
    const uint32_t xbytes = (uint32_t)KT * 512u;  // tokens: [K step][4][128 bytes], 16-byte chunk c of token r at position c ^ 2 r; their scales behind them
    uint8_t* const own = smem + xbytes + 256 + wave * D * STAGE;
    auto dma_w = [&](int kt, int st) {
        uint8_t* const to = own + st * STAGE;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool in = MX ? few_codes_inside(kt, chunk[h], (uint32_t)p.K) : kt < KT;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_void*)(to + h * 1024), 16, in ? vw[h] : kOutside, (uint32_t)kt << (MX ? 6 : 7), 0, 2);
        }
        if (MX) {
            const int ks = kt + ((lane >> 4) & 1);
            const uint32_t at = lane < 32 && ks < KT ? (uint32_t)lrow * (uint32_t)p.ld_ws + ((uint32_t)ks << 2) : kOutside;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsc, (lds_void*)(to + 2048), 4, at, 0, 0, 0);
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) dma_w(d * WK, d);
    if (wave < p.M) {
        u32 m = 0;
#pragma unroll
        for (int j = 0; j < V; ++j) m = absmax8(m, v[j]);
        const float scale = scale_from_amax(amax_from_bits(wave_max(pk_fold(m))));
        const Divider dv(scale);
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const int i = lane + 64 * j;
            const uint2 q = cast8(v[j], dv);
            const uint32_t at = (uint32_t) reinterpret_cast<uintptr_t>((lds_void*)(smem + (i >> 4) * 512 + wave * 128 + ((((i & 15) >> 1) ^ (wave << 1)) << 4) + (i & 1) * 8));
            const uint64_t both = (uint64_t)q.x | ((uint64_t)q.y << 32);
            // (LDS by instructions written out: in front of a store it knows of, the compiler waits for every load in flight)
            if (i < nvec) asm volatile("ds_write_b64 %0, %1" ::"v"(at), "v"(both) : "memory");
        }
        const uint32_t at = (uint32_t) reinterpret_cast<uintptr_t>((lds_void*)(smem + xbytes + wave * 4));
        if (lane == 0) asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(scale) : "memory");
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    const int fr = (((lrow >> 1) & 1) << F1) | (((lrow >> 3) & 1) << 2), c0 = MX ? quarter : 2 * quarter, other = MX ? 64 : 16;
    const int fo = lrow * 128 + ((c0 ^ fr) << 4), token = lrow & 3;  // (the lanes of tokens that there are not read another one or what LDS held, for columns that are not stored)
    const int xo = token * 128 + ((c0 ^ (token << 1)) << 4);
    auto two = [&](const uint8_t* at, int o) {
        const i32x4 lo = *reinterpret_cast<const i32x4*>(at + o);
        const i32x4 hi = *reinterpret_cast<const i32x4*>(at + (o ^ other));
        return i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    f32x4 acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    int st = 0;
    for (int k0 = 0; k0 < KT; k0 += 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = k0 + j, s = j % WK;
            if (k < KT) {
                if (s == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(WL * (D - 1)) : "memory");
                const uint8_t* const at = own + st * STAGE;
                i32x8 w;
                int wsc = 0;
                if (MX) {
                    const i32x4 a = *reinterpret_cast<const i32x4*>(at + (fo ^ (s * 64)));
                    w = i32x8{a[0], a[1], a[2], a[3], 0, 0, 0, 0};
                    wsc = (int)(*reinterpret_cast<const u32*>(at + 2048 + s * 64 + lrow * 4) >> (quarter * 8));
                } else {
                    w = two(at, fo);
                }
                const i32x8 xf = two(smem + k * 512, xo);
                if (MX) acc[j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, xf, acc[j], 4, 0, 0, wsc, 0, 0x7F7F7F7F);
                else acc[j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, xf, acc[j], 0, 0, 0, 0, 0, 0);
                asm volatile("" : "+v"(acc[j]));  // the fragments have been read
                CFP8_PHASE_END();
                if (s == WK - 1 || k == KT - 1) {
                    dma_w(k + 1 + (D - 1) * WK, st);
                    st = st == D - 1 ? 0 : st + 1;
                }
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may land in LDS once the workgroup has gone
    const int n = nw0 + quarter * 4;
    if (n >= p.N || lrow >= p.M) return;
    const float sam = *reinterpret_cast<const float*>(smem + xbytes + lrow * 4);
    const f32x4 sbn = MX ? f32x4{1.f, 1.f, 1.f, 1.f} : *reinterpret_cast<const f32x4*>(p.sb + n);
    const uint2 bia = p.bias ? *reinterpret_cast<const uint2*>(p.bias + n) : make_uint2(kNoBias, kNoBias);
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (((acc[0][e] + acc[1][e]) + acc[2][e]) + acc[3][e]) * sam * sbn[e];
    if (f32) {
        *reinterpret_cast<f32x4*>(static_cast<float*>(p.out) + (int64_t)lrow * p.ld_out + n) = plus_bias<true>(o, bia.x, bia.y);
    } else {
        o = plus_bias<false>(o, bia.x, bia.y);
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.out) + (int64_t)lrow * p.ld_out + n) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
    }
}

template <int MODE, int V>
static int launch_linear_stream_cfg(const RingArgs& p, const void* x, int64_t ld_x, int waves, int out_dtype, hipStream_t st) {
    const size_t lds = (size_t)(p.K >> 7) * 512 + 256 + (size_t)waves * few_depth(MODE, 1) * few_stage(MODE);
    auto* const kern = linear_stream_kernel<MODE, V>;
    static std::atomic<bool> raised[65];
    const int slot = device_slot();
    if (slot == 64) raised[64].store(false, std::memory_order_relaxed);
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kern), 160 * 1024, raised[slot])) return rc;
    const unsigned blocks = (unsigned)((p.N / 16 + waves - 1) / waves);
    if (!note_launch(MODE == kRingMx ? "linear_mxfp4_stream" : "linear_stream", blocks, (unsigned)waves * 64, lds)) return CFP8_OK;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3((unsigned)waves * 64), lds, st, p, static_cast<const uint4*>(x), ld_x / 8, (int)(out_dtype == CFP8_OUT_F32));
    return check_launch("linear");
}

template <int MODE, int TM, int WIDTH>
static int launch_few_cfg(RingArgs& p, int waves, size_t scales, int out_dtype, const char* name, hipStream_t st) {
    using Sh = FewShape<MODE, TM, WIDTH>;
    if (waves < Sh::LEAST || waves * 64 > few_threads(WIDTH)) return set_error(CFP8_EINVAL, "gemm: %d strips of %d rows have no form", waves, p.M);
    const size_t lds = Sh::WB + (size_t)waves * Sh::WS + scales;
    auto* const kern = gemm_ring_few_kernel<MODE, TM, WIDTH>;
    static std::atomic<bool> raised[65];
    const int slot = device_slot();
    if (slot == 64) raised[64].store(false, std::memory_order_relaxed);
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kern), 160 * 1024, raised[slot])) return rc;
    const unsigned blocks = (unsigned)(p.tiles_n * p.slices);
    if (note_launch(name, blocks, (unsigned)waves * 64, lds)) hipLaunchKernelGGL(kern, dim3(blocks), dim3((unsigned)waves * 64), lds, st, p, (int)(out_dtype == CFP8_OUT_F32));
    return CFP8_OK;
}
template <int MODE, int TM>
static int launch_few_tm(RingArgs& p, int strips, size_t scales, int out_dtype, const char* name, hipStream_t st) {
    if constexpr (TM > 1) {
        if (p.M <= 16 * (TM - 1)) return launch_few_tm<MODE, TM - 1>(p, strips, scales, out_dtype, name, st);
    }
    if constexpr (TM <= 2) {
        if (strips < 4) return launch_few_cfg<MODE, TM, 0>(p, strips, scales, out_dtype, name, st);
    }
    if constexpr (TM <= (MODE == kRingRow ? 5 : 8)) {
        if (strips < 8) return launch_few_cfg<MODE, TM, 1>(p, strips, scales, out_dtype, name, st);
    }
    return launch_few_cfg<MODE, TM, 2>(p, strips, scales, out_dtype, name, st);
}

// bytes of LDS that the scales of a block-scaled workgroup of `waves` strips take
static size_t few_scales(const RingArgs& p, int waves) {
    const int steps = p.slice_steps, blocks = (waves * 16 + 111) / 128 + 1;
    return (size_t)(((p.M * (steps | 1) + 63) & ~63) + blocks * ((steps + 63) & ~63)) * 4;
}
// Whether LDS holds what a workgroup of `strips` needs, and 32-bit offsets reach the weight scales.
static bool few_fits(int mode, const RingArgs& p, int strips) {
    if (mode == kRingBlock && ((p.N + 127) / 128 * p.sb_stride_n + (p.K >> 7) * p.sb_stride_k) * 4 >= ((int64_t)1 << 31)) return false;
    const int tm = (p.M + 15) / 16;
    const size_t x = (size_t)few_chunks(tm) * few_steps(tm) * tm * 2048 + 1024, scales = mode == kRingBlock ? few_scales(p, strips) : 0;
    return strips <= 12 && x + scales + (size_t)strips * few_depth(mode, tm) * few_stage(mode) <= 160 * 1024;
}

}  // namespace cfp8
