// Device code of the small bf16 tiles (gemm.hip, gemm_pairs.hip): the
// activation stage and the stores of a tile.
#pragma once

#include "gemm_common.h"

namespace srq {
namespace {

constexpr int XLD = 72;

template <int TM, int NT = 256>
struct XTile {
    static constexpr int BM = TM * 16;
    static constexpr int FPT = BM * 64 / NT;  // staged floats per thread (16, 8 or 4)
    static constexpr int TPR = 64 / FPT;      // threads per row
    static constexpr int NV = FPT / 4;
    static constexpr int PLANE = BM * XLD;    // bf16 per plane
    static_assert(FPT >= 4, "at least one float4 per thread");
};

// Splits the staged floats into the hi / mid / lo planes; returns max |x|.
template <int TM, int NT = 256>
__device__ __forceinline__ float xstore_a(__bf16 *As, int tid, const float4 (&a)[XTile<TM, NT>::NV]) {
    typedef XTile<TM, NT> X;
    constexpr int FPT = X::FPT, TPR = X::TPR, NV = X::NV, PLANE = X::PLANE;
    const int r = tid / TPR, c = (tid % TPR) * FPT;
    float amax = 0.0f;
    uint32_t ph[FPT / 2], pm[FPT / 2], pl[FPT / 2];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const float v[4] = {a[i].x, a[i].y, a[i].z, a[i].w};
        float r1[4], r2[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            amax = fmaxf(amax, fabsf(v[e]));
            r1[e] = v[e] - __uint_as_float(__float_as_uint(v[e]) & 0xFFFF0000u);
            r2[e] = r1[e] - __uint_as_float(__float_as_uint(r1[e]) & 0xFFFF0000u);
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            ph[2 * i + e] = pk_hi16(v[2 * e], v[2 * e + 1]);
            pm[2 * i + e] = pk_hi16(r1[2 * e], r1[2 * e + 1]);
            pl[2 * i + e] = pk_hi16(r2[2 * e], r2[2 * e + 1]);
        }
    }
    __bf16 *dst = As + r * XLD + c;
    if constexpr (FPT == 4) {
        *(uint2 *)dst = make_uint2(ph[0], ph[1]);
        *(uint2 *)(dst + PLANE) = make_uint2(pm[0], pm[1]);
        *(uint2 *)(dst + 2 * PLANE) = make_uint2(pl[0], pl[1]);
    } else {
#pragma unroll
        for (int i = 0; i < FPT / 8; ++i) {
            *(uint4 *)(dst + 8 * i) = make_uint4(ph[4 * i], ph[4 * i + 1], ph[4 * i + 2], ph[4 * i + 3]);
            *(uint4 *)(dst + PLANE + 8 * i) = make_uint4(pm[4 * i], pm[4 * i + 1], pm[4 * i + 2], pm[4 * i + 3]);
            *(uint4 *)(dst + 2 * PLANE + 8 * i) = make_uint4(pl[4 * i], pl[4 * i + 1], pl[4 * i + 2], pl[4 * i + 3]);
        }
    }
    return amax;
}

// Stores a tile's accumulators: partial sums of its K slice (partial !=
// nullptr), else y (+ residual), rows holding a |x| > kWideLimit recomputed
// in FP64.  D layout of 16x16x32: lane holds rows 4*(lane/16)+r, column
// lane%16.
// TN feature tiles per wave, XBN features and NT threads per workgroup.
template <int TM, int TN, int XBN = 64 * TN, int NT = 256>
__device__ __forceinline__ void x3_finish(const GemmArgs &G, float *__restrict__ partial, int32_t *__restrict__ wflags,
                                          const floatx4 (&acc)[TM][TN], const float amax, int *row_wide,
                                          const int64_t n0, const int64_t m0, const int tid) {
    constexpr int BM = XTile<TM>::BM;
    const int lane = tid & 63, li = lane & 15, q = lane >> 4;
    if (amax > kWideLimit) row_wide[tid / XTile<TM, NT>::TPR] = 1;
    lds_barrier();

    if (partial) {
        float *P = partial + (int64_t)blockIdx.z * G.n * G.rows;
        if (blockIdx.x == 0 && tid < BM && m0 + tid < G.n) wflags[(int64_t)blockIdx.z * G.n + m0 + tid] = row_wide[tid];
        const int64_t nw = (int64_t)blockIdx.x * XBN;  // the workgroup's first feature
        if (m0 + BM <= G.n && nw + XBN <= G.rows && G.rows * BM < (int64_t(1) << 30)) {
            // Every output of the workgroup is in bounds (a uniform test) and
            // its byte offsets from the corner fit 32 bits: no per-store checks.
            float *Pt = P + m0 * G.rows + nw;
            const uint32_t ld = (uint32_t)G.rows, c0 = (uint32_t)(n0 - nw) + (uint32_t)li;
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t mo = (uint32_t)(tm * 16 + 4 * q + r) * ld + c0;
#pragma unroll
                    for (int tn = 0; tn < TN; ++tn)
                        *(float *)((char *)Pt + (mo + (uint32_t)(tn * 16)) * 4u) = acc[tm][tn][r];
                }
            return;
        }
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t m = m0 + tm * 16 + 4 * q + r;
                if (m >= G.n) continue;
#pragma unroll
                for (int tn = 0; tn < TN; ++tn) {
                    const int64_t j = n0 + tn * 16 + li;
                    if (j < G.rows) P[m * G.rows + j] = acc[tm][tn][r];
                }
            }
        return;
    }
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int mi = tm * 16 + 4 * q + r;
            const int64_t m = m0 + mi;
            if (m >= G.n || row_wide[mi]) continue;
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) {
                const int64_t j = n0 + tn * 16 + li;
                if (j >= G.rows) continue;
                float v = acc[tm][tn][r];
                if (G.residual) v = G.residual[m * G.y_stride + j] + v;
                G.y[m * G.y_stride + j] = v;
            }
        }
    for (int mi = 0; mi < BM; ++mi) {
        if (!row_wide[mi] || m0 + mi >= G.n) continue;
        const int64_t j = (int64_t)blockIdx.x * XBN + tid;
        if (tid < XBN && j < G.rows) G.y[(m0 + mi) * G.y_stride + j] = wide_output(G, m0 + mi, j);
    }
}

}  // namespace
}  // namespace srq
