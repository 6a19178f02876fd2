// Device code shared by the GEMM kernels (gemm.hip, gemm_tall.hip, gemm_f32.hip).
#pragma once

#include "srq_internal.h"

namespace srq {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

// linearQ8WideInto / linearQ4WideInto (M:4356-4382, M:4754-4780): output o
// of row m in FP64, per-block partial sums scaled in FP64, plus residual.
__device__ __forceinline__ double wide_weight(int fmt, const uint8_t *wrow, int64_t c) {
    if (fmt == SRQ_Q8) return (double)((const int8_t *)wrow)[c];
    if (fmt == SRQ_Q4) {
        uint32_t b = wrow[c >> 1];
        uint32_t nib = (c & 1) ? (b >> 4) : (b & 15u);
        return (double)(((int32_t)(nib << 28)) >> 28);
    }
    return (double)((const float *)wrow)[c];
}

__device__ __forceinline__ float wide_output(const GemmArgs &G, int64_t m, int64_t o) {
    const uint8_t *wrow = (const uint8_t *)G.values + o * row_bytes(G.fmt, G.cols);
    const float *xr = G.x + m * G.cols;
    const int64_t groups = groups_of(G.cols);
    double sum = 0.0;
    for (int64_t g = 0; g < groups; ++g) {
        double part = 0.0;
        const int64_t end = (g + 1) * kBlock < G.cols ? (g + 1) * kBlock : G.cols;
        for (int64_t j = g * kBlock; j < end; ++j) part += (double)xr[j] * wide_weight(G.fmt, wrow, j);
        sum += part * (G.fmt == SRQ_F32 ? 1.0 : (double)G.scales[o * groups + g]);
    }
    float v = (float)sum;
    if (G.residual) v = G.residual[m * G.y_stride + o] + v;
    return v;
}

// Stores a workgroup's MFMA tiles: partial sums of its K slice (partial !=
// nullptr; wide-row flags from the first feature tile), else y (+ residual),
// rows holding a |x| > kWideLimit recomputed in FP64.  D layout of the 16x16
// MFMAs: lane holds rows 4*(lane/16)+r, column lane%16.  BM rows x BN features
// from (m0, n0); this wave's TM x TN tiles start at (mw, nw) of them.
template <int BM, int BN, int TM, int TN>
__device__ __forceinline__ void gemm_finish(const GemmArgs &G, float *__restrict__ partial,
                                            int32_t *__restrict__ wflags, const floatx4 (&acc)[TM][TN],
                                            const int *row_wide, const int64_t n0, const int64_t m0, const int mw,
                                            const int nw, const int tid) {
    const int li = tid & 15, gq = (tid & 63) >> 4;
    if (partial) {
        float *P = partial + (int64_t)blockIdx.z * G.n * G.rows;
        if (blockIdx.x == 0 && tid < BM && m0 + tid < G.n) wflags[(int64_t)blockIdx.z * G.n + m0 + tid] = row_wide[tid];
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t m = m0 + mw + tm * 16 + 4 * gq + r;
                if (m >= G.n) continue;
#pragma unroll
                for (int tn = 0; tn < TN; ++tn) {
                    const int64_t j = n0 + nw + tn * 16 + li;
                    if (j < G.rows) P[m * G.rows + j] = acc[tm][tn][r];
                }
            }
        return;
    }
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int mi = mw + tm * 16 + 4 * gq + r;
            const int64_t m = m0 + mi;
            if (m >= G.n || row_wide[mi]) continue;
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) {
                const int64_t j = n0 + nw + tn * 16 + li;
                if (j >= G.rows) continue;
                float v = acc[tm][tn][r];
                if (G.residual) v = G.residual[m * G.y_stride + j] + v;
                G.y[m * G.y_stride + j] = v;
            }
        }
    // This workgroup saw all of K: it recomputes its wide rows itself.
    for (int mi = 0; mi < BM; ++mi) {
        if (!row_wide[mi] || m0 + mi >= G.n) continue;
        const int64_t j = n0 + tid;
        if (tid < BN && j < G.rows) G.y[(m0 + mi) * G.y_stride + j] = wide_output(G, m0 + mi, j);
    }
}

// Workgroup barrier over LDS only.  __syncthreads() also waits for every
// global load in flight (vmcnt(0)), which in the block loop below would
// drain the weight and activation loads issued blocks ahead at every block.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// LDS-direct loads: 16 (4) bytes per lane from base + voff (32-bit, per lane)
// to lds + 16 (4) * lane.  In asm because the compiler would make every later
// LDS read wait for them; the block loop waits for them itself.
__device__ __forceinline__ void lds_load16(uint32_t lds, uint32_t voff, const uint8_t *base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds), "v"(voff), "s"(base)
                 : "memory");
}
__device__ __forceinline__ void lds_load4(uint32_t lds, uint32_t voff, const uint8_t *base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :
                 : "s"(lds), "v"(voff), "s"(base)
                 : "memory");
}
// The same 16 bytes from an address per lane.
__device__ __forceinline__ void lds_load16(uint32_t lds, const uint8_t *p) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds), "v"(p) : "memory");
}

__device__ __forceinline__ uint32_t pk_hi16(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

// One lane's 16 codes of a block: Q8 16 bytes, Q4 8 bytes.
template <int FMT>
struct XRaw {
    typedef uint32_t type __attribute__((ext_vector_type(FMT == SRQ_Q8 ? 4 : 2)));
};

// Codes of one lane's block slice -> the two bf16x8 MFMA operands.
template <int FMT>
__device__ __forceinline__ void xcodes(const typename XRaw<FMT>::type raw, bf16x8 &h0, bf16x8 &h1) {
    u32x4v p0, p1;
    if constexpr (FMT == SRQ_Q8) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const uint32_t d = raw[w];
            const float c0 = (float)(int32_t)(int8_t)d, c1 = (float)(int32_t)(int8_t)(d >> 8);
            const float c2 = (float)(int32_t)(int8_t)(d >> 16), c3 = (float)((int32_t)d >> 24);
            const uint32_t a = pk_hi16(c0, c1), b = pk_hi16(c2, c3);
            if (w < 2) {
                p0[2 * w] = a;
                p0[2 * w + 1] = b;
            } else {
                p1[2 * w - 4] = a;
                p1[2 * w - 3] = b;
            }
        }
    } else {
        // code/16 (exact in bf16), one SDWA convert per nibble; the block's
        // scale carries the factor 16 back (SRQ_CONVERT), so the product
        // block * scale is unchanged bit for bit
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const uint32_t d = raw[w], h = d >> 4;
            u32x4v &p = w == 0 ? p0 : p1;
            p[0] = pk_hi16(nib16<0>(d), nib16<0>(h));
            p[1] = pk_hi16(nib16<1>(d), nib16<1>(h));
            p[2] = pk_hi16(nib16<2>(d), nib16<2>(h));
            p[3] = pk_hi16(nib16<3>(d), nib16<3>(h));
        }
    }
    h0 = __builtin_bit_cast(bf16x8, p0);
    h1 = __builtin_bit_cast(bf16x8, p1);
}

}  // namespace

constexpr int64_t kTallMaxCols = int64_t(1) << 22;

// gemm_tall.hip: a wave's 16-row tiles and the waves per workgroup.
struct TallPlan {
    int tm, nw;
};
TallPlan tall_plan(int32_t n, int64_t rows, int slices);
// Bytes of the activations' bf16 planes.
size_t tall_plane_bytes(const TallPlan &p, int32_t n, int64_t cols);
// wflags: slices * n words; partial as gemm_x3_kernel's (null: writes y).
int launch_gemm_tall(hipStream_t s, const GemmArgs &a, const TallPlan &p, uint8_t *planes, float *partial,
                     int32_t *wflags, int slices, int kper);

// gemm_pairs.hip: calls of at most 32 rows (bm 16 or 32, tn as plan_gemm's)
// whose weights it can read by 128-byte row segments.
bool gemm_pairs_ok(const GemmArgs &a, int kper);
void launch_gemm_pairs(hipStream_t s, const GemmArgs &a, int bm, int tn, float *partial, int32_t *wflags, int slices,
                       int kper);

// gemm_f32.hip: F32 weights, cols % 32 == 0; kper counts K steps of 32.
int launch_gemm_f32(hipStream_t s, const GemmArgs &a, float *partial, int32_t *wflags, int slices, int kper);

}  // namespace srq
