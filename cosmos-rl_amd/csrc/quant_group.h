// The 1x128 group quantiser of activations, for the kernels that run it: alone, or beside the routing of a MoE layer's tokens.
#pragma once

#include "cfp8_common.h"

namespace cfp8 {

constexpr int64_t kMaxGroups = 0xFFFFFF00ll;

struct GroupRows {
    const uint4* x;   // bf16 rows
    uint2* q;         // fp8 rows
    float* scales;    // [rows, ngroups]
    int64_t ldx, ldq; // in vectors of 8 values
    int nvec;         // vectors a row
    u32 ngroups, rows, total_groups;
};
inline GroupRows group_rows(const void* x, int64_t rows, int64_t cols, int64_t ld_x, void* q, int64_t ld_q, float* scales) {
    const int64_t ngroups = (cols + 127) / 128;
    return {static_cast<const uint4*>(x), static_cast<uint2*>(q), scales, ld_x / 8, ld_q / 8, (int)(cols / 8), (u32)ngroups, (u32)rows, (u32)(rows * ngroups)};
}

// ---------------------------------------------------------------------------
// 1x128 groups.  16 lanes own one group (one 16-byte vector each), the max runs
// over the 16-lane DPP row.  Every thread handles N groups that follow each other: 4 so that four loads are in flight
// per lane, 1 where there are so few groups that a thread's casts, one behind the other, are what takes the time.
// ---------------------------------------------------------------------------
// With GATHER, output row r quantises input row src_rows[r] (a zero row where that is negative): the token
// gather in front of the grouped GEMM and the quantiser in one pass, without the gathered bf16 matrix.
// Groups are numbered row-major (row * ngroups + column) in 32 bits; a thread divides once and steps
// through its consecutive groups.  Every load is unconditional on a clamped address (what must read
// as zero is cleared afterwards), so all are in flight before the first is used.
template <int MODE, int N, bool GATHER = false>
__device__ __forceinline__ void group128_some(const GroupRows& p, u32 g0, const int32_t* __restrict__ src_rows = nullptr) {
    const int sub = threadIdx.x & 15;
    const u32 ngroups = p.ngroups, rows = p.rows, total_groups = p.total_groups;
    const int nvec = p.nvec;
    const int64_t ldx = p.ldx, ldq = p.ldq;
    const uint4* __restrict__ const x = p.x;
    uint2* __restrict__ const q = p.q;
    float* __restrict__ const scales = p.scales;
    uint4 v[N];
    u32 row[N], gcol[N];
    bool ok[N];
    {
        u32 r = g0 / ngroups, c = g0 - r * ngroups;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            row[i] = r;
            gcol[i] = c;
            if (++c == ngroups) c = 0, ++r;
        }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int vec = (int)gcol[i] * 16 + sub;
        ok[i] = g0 + i < total_groups && vec < nvec;
        const u32 rc = row[i] < rows ? row[i] : rows - 1;
        const int vc = vec < nvec ? vec : nvec - 1;
        if (GATHER) {
            const int32_t src = src_rows[rc];
            ok[i] = ok[i] && src >= 0;
            // tokens are read several times (once per expert they go to): leave them in the caches
            v[i] = ld16<false>(x + (int64_t)(src >= 0 ? src : 0) * ldx + vc);
        } else {
            v[i] = ld16<true>(x + (int64_t)rc * ldx + vc);
        }
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (!ok[i]) v[i] = make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const u32 m = row16_max(pk_fold(absmax8(0u, v[i])));
        const float amax = amax_from_bits(m);
        uint2 out;
        float scale;
        if (MODE == CFP8_GROUP_MODE_DIV) {
            scale = scale_from_amax(amax);
            const Divider d(scale);
            out = cast8(v[i], d);
        } else {
            // x * (448 / clamp(amax, 1e-4)) as torch evaluates `448.0 / tensor`:
            // reciprocal first, then times 448.  No clamp before the cast: the product
            // exceeds 448 by at most a few fp32 roundings, far below the NaN threshold 464
            if (amax != amax) {
                scale = __uint_as_float(kCanonNaN);
                out = make_uint2(0x7F7F7F7Fu, 0x7F7F7F7Fu);
            } else {
                const float a = fmaxf(amax, 1e-4f);
                const float mul = (1.0f / a) * kE4M3Max;
                scale = a / kE4M3Max;
                const u32 w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
                u32 o[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    u32 p = cvt2<false>(bf16_lo(w[2 * k]) * mul, bf16_hi(w[2 * k]) * mul, 0u);
                    o[k] = cvt2<true>(bf16_lo(w[2 * k + 1]) * mul, bf16_hi(w[2 * k + 1]) * mul, p);
                }
                out = make_uint2(o[0], o[1]);
            }
        }
        const int vec = (int)gcol[i] * 16 + sub;
        if (g0 + i < total_groups && vec < nvec) q[(int64_t)row[i] * ldq + vec] = out;
        if (sub == 0 && g0 + i < total_groups) scales[g0 + i] = scale;
    }
}

}  // namespace cfp8
