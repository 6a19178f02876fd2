// Dequant-GEMM for prefill chunks: Q8 / Q4 weights, many activation rows.
//
// The arithmetic is gemm_x3_kernel's (gemm.hip): three exact bf16 terms per
// activation, six v_mfma_f32_16x16x32_bf16 per 16x16x64 block from zero in
// the same order, then acc = fma(block, scale, acc); every output has the
// same bits.  What differs is who does the work around the MFMAs, which took
// most of gemm_x3_kernel's time (MFMA pipe busy 37% at 28672 x 4096 Q4, 256
// rows):
//  - The activations are split into their bf16 planes once per call
//    (gemm_split_kernel), not once per workgroup and block.  The planes are
//    stored as the LDS images the GEMM stages, so a block's stage is a plain
//    copy by LDS-direct loads: no VALU work, no registers, no LDS writes by
//    the wave.
//  - A wave owns up to 128 rows x 64 features, so each converted weight
//    feeds up to eight row tiles.
//  - Scales come four blocks at a time, and the weights' cache lines are
//    touched blocks ahead, a share of the rows per block.
//  - The scale FMAs issue between the next tile's MFMAs, and a wave inside
//    its MFMA steps outranks its SIMD's other wave.
// Measured, whole srq_linear call, gemm_x3_kernel -> here: 28672 x 4096 Q4 at
// 256 rows 194 -> 151 us, 4096 x 14336 Q8 at 1000 rows 370 -> 316 us.  What
// bounds it: the MFMAs and their operand reads alone take 100 of the 130 us the
// first case's GEMM takes, code conversion, scale FMAs and loads the rest.
#include <algorithm>

#include "gemm_common.h"

namespace srq {
namespace {

constexpr int kSplitThreads = 256;
constexpr int kRowBytes = kBlock * 2;  // one row of one plane's image

// Image of row tile rt and block g: [plane hi, mid, lo][row][8 chunks of 16
// bytes], chunk c of row r at slot c ^ (r % 8), so that an operand read of
// one chunk of 16 rows touches every bank once.  Row m of x: one workgroup.
__global__ __launch_bounds__(kSplitThreads) void gemm_split_kernel(const float *__restrict__ x, const int64_t cols,
                                                                   const int32_t n, const int bm, const int slices,
                                                                   uint8_t *__restrict__ planes,
                                                                   int32_t *__restrict__ wflags) {
    const int64_t m = blockIdx.x, groups = cols / kBlock;
    const int64_t rt = m / bm;
    const int r = (int)(m - rt * bm);
    const int plane = bm * kRowBytes;
    const float *xr = x + m * cols;
    uint8_t *out = planes + rt * groups * 3 * plane + r * kRowBytes;
    float amax = 0.0f;
    for (int64_t i = threadIdx.x; i < cols / 8; i += kSplitThreads) {
        const float4 a = *(const float4 *)(xr + 8 * i), b = *(const float4 *)(xr + 8 * i + 4);
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        uint32_t h[4], d[4], l[4];
        float r1[8], r2[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            amax = fmaxf(amax, fabsf(v[e]));
            r1[e] = v[e] - __uint_as_float(__float_as_uint(v[e]) & 0xFFFF0000u);
            r2[e] = r1[e] - __uint_as_float(__float_as_uint(r1[e]) & 0xFFFF0000u);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            h[e] = pk_hi16(v[2 * e], v[2 * e + 1]);
            d[e] = pk_hi16(r1[2 * e], r1[2 * e + 1]);
            l[e] = pk_hi16(r2[2 * e], r2[2 * e + 1]);
        }
        uint8_t *dst = out + (i >> 3) * 3 * plane + (((int)i & 7) ^ (r & 7)) * 16;
        *(uint4 *)dst = make_uint4(h[0], h[1], h[2], h[3]);
        *(uint4 *)(dst + plane) = make_uint4(d[0], d[1], d[2], d[3]);
        *(uint4 *)(dst + 2 * plane) = make_uint4(l[0], l[1], l[2], l[3]);
    }
    const int wide = __syncthreads_or(amax > kWideLimit);
    for (int z = threadIdx.x; z < slices; z += kSplitThreads) wflags[(int64_t)z * n + m] = wide;
}

// lds_load16 unless `skip` (uniform) is not 0.  The branch is inside the asm:
// around it, the compiler would keep two copies of the accumulators.
__device__ __forceinline__ void lds_load16_unless(uint32_t skip, uint32_t lds, uint32_t voff, const uint8_t *base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_cmp_lg_u32 %3, 0\n\ts_cbranch_scc1 .Lskip%=\n\t"
                 "global_load_lds_dwordx4 %1, %2\n.Lskip%=:"
                 :
                 : "s"(lds), "v"(voff), "s"(base), "s"(__builtin_amdgcn_readfirstlane(skip))
                 : "memory", "scc");
}

// s_waitcnt vmcnt(N), the other counters unconstrained.  The builtin, so that
// the compiler knows its own loads have landed and adds no wait for them.
template <int N>
__device__ __forceinline__ void wait_loads() {
    static_assert(N < 16, "vmcnt's low field");
    __builtin_amdgcn_s_waitcnt(0x0F70 | N);
    asm volatile("" ::: "memory");
}

constexpr int kScaleGroup = 4;  // blocks whose scales one load brings

// TM 16-row tiles and 64 features per wave, NW waves (64 * NW features) per
// workgroup.  kper counts 64-input blocks; slices as in gemm_x3_kernel.
// cols % 256 == 0 (16-byte scale loads) and cols <= kTallMaxCols (32-bit
// offsets within a workgroup's rows).
template <int FMT, int TM, int NW>
__global__ __launch_bounds__(64 * NW, 2) void gemm_tall_kernel(const GemmArgs G, const uint8_t *__restrict__ planes,
                                                               float *__restrict__ partial,
                                                               const int32_t *__restrict__ wflags, const int kper) {
    constexpr int TN = 4, BM = 16 * TM, XBN = 64 * NW;
    constexpr int PLANE = BM * kRowBytes, IMAGE = 3 * PLANE, LOADS = IMAGE / 1024;
    constexpr uint32_t BB = FMT == SRQ_Q8 ? kBlock : kBlock / 2;  // weight bytes per row and block
    typedef typename XRaw<FMT>::type R;
    __shared__ __attribute__((aligned(16))) uint8_t As[2][IMAGE];
    __shared__ __attribute__((aligned(16))) float Ss[NW][2][64 * kScaleGroup];
    __shared__ uint32_t sink[NW][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, q = lane >> 4;
    const int64_t nw = (int64_t)blockIdx.x * XBN, m0 = (int64_t)blockIdx.y * BM;
    const int groups = (int)(G.cols / kBlock);
    const int gbeg = (int)blockIdx.z * kper;
    const int gend = min(gbeg + kper, groups);

    // 32-bit offsets from the workgroup's first feature row; rows past the
    // end read row rows-1 and are never stored
    const uint8_t *wb = (const uint8_t *)G.values + nw * groups * BB;
    const uint8_t *sb = (const uint8_t *)(G.scales + nw * groups);
    uint32_t wo[TN];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
        const int64_t row = min(nw + wave * 64 + tn * 16 + li, G.rows - 1) - nw;
        wo[tn] = (uint32_t)(row * groups * BB) + (BB / 4) * q;
    }
    const uint32_t lrow = (uint32_t)(min(nw + wave * 64 + lane, G.rows - 1) - nw);  // this lane's row of the wave's 64
    const uint8_t *img = planes + ((int64_t)blockIdx.y * groups + gbeg) * IMAGE;
    const uint32_t as0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)&As[0][0];
    const uint32_t sink0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t *)&sink[wave][0];
    auto stage = [&](const uint32_t at) {
#pragma unroll
        for (int k = 0; k < (LOADS + NW - 1) / NW; ++k) {
            const int c = k * NW + wave;
            if (LOADS % NW == 0 || c < LOADS)
                lds_load16(as0 + at + (uint32_t)(c * 1024), (uint32_t)(lane * 16), img + c * 1024);
        }
    };

    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    R raw[TN];
    auto load_w = [&](const int g) {
        const uint8_t *w = wb + (uint32_t)g * BB;
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) raw[tn] = *(const R *)(w + (uint64_t)wo[tn]);
    };
    // The scales of the wave's 64 rows, lane = row: four blocks (4k .. 4k+3 of
    // the matrix) in one load, into Ss[wave][k & 1][row][block].  Loads of
    // one block's scales of 16 rows each would cost a cache-line request per
    // row and block; these cost one per row and four blocks.
    const uint32_t ss0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float *)&Ss[wave][0][0];
    const uint32_t so = lrow * (uint32_t)groups * 4u;
    auto load_s = [&](const int skip, const int k) {
        lds_load16_unless((uint32_t)skip, ss0 + (uint32_t)(k & 1) * 64 * kScaleGroup * 4, so,
                      sb + (uint32_t)min(k * kScaleGroup, groups - kScaleGroup) * 4);
    };
    // Touch of the cache lines of the weights LB..2*LB blocks on (a line
    // holds LB blocks of a row), 64 / LB rows per block, so that the loads that
    // need them find them in L2: all workgroups walk K together, and without
    // it every LBth block waits for one line of every row at once.
    constexpr int LB = 128 / BB;
    const uint32_t trow = (uint32_t)(wave * 64 + (lane & ~(LB - 1)));
    const uint32_t tlast = (uint32_t)min((int64_t)XBN, G.rows - nw) - 1;
    auto touch = [&](const int g) {
        lds_load4(sink0, min(trow + (uint32_t)(g & (LB - 1)), tlast) * ((uint32_t)groups * BB),
                  wb + (uint32_t)min((g / LB + 2) * LB, groups - 1) * BB);
    };
    load_s(0, gbeg / kScaleGroup);
    load_w(gbeg);
    stage(0);
    wait_loads<0>();
    lds_barrier();

    // operand chunk of half h in row li of a tile: 2q + h, swizzled
    const int rd[2] = {((2 * q) ^ (li & 7)) * 16 + li * kRowBytes, ((2 * q + 1) ^ (li & 7)) * 16 + li * kRowBytes};
    uint32_t cur = 0;  // byte offset of the block's stage
    for (int g = gbeg; g < gend; ++g) {
        // the next block's loads (the last block loads itself again)
        const int next = min(g + 1, gend - 1);
        img += (next - g) * IMAGE;
        stage(IMAGE - cur);
        load_s(next % kScaleGroup, next / kScaleGroup);
        touch(g);
        bf16x8 b[TN][2];
        float s[TN];
        const float *sl = &Ss[wave][(g / kScaleGroup) & 1][g % kScaleGroup];
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
            xcodes<FMT>(raw[tn], b[tn][0], b[tn][1]);
            const float sc = sl[(tn * 16 + li) * kScaleGroup];
            s[tn] = FMT == SRQ_Q4 ? 16.0f * sc : sc;
        }
        load_w(next);
        // Steps (tm, plane): a step's two operands are read one step ahead, and
        // a row tile's sums are scaled in during the next tile's first step.
        // sched_barrier keeps the steps apart: without it the scheduler hoists
        // operand reads of several tiles and spills.
        const uint8_t *as = &As[0][0] + cur;
        bf16x8 a[2][2];
        floatx4 blk[2][TN];
        auto read = [&](const int step) {
            const int tm = step / 3, t = 2 - step % 3;
#pragma unroll
            for (int h = 0; h < 2; ++h)
                a[step & 1][h] = *(const bf16x8 *)(as + t * PLANE + tm * 16 * kRowBytes + rd[h]);
        };
        auto scale = [&](const int tm) {
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc[tm][tn][r] = __builtin_fmaf(blk[tm & 1][tn][r], s[tn], acc[tm][tn][r]);
        };
        __builtin_amdgcn_s_setprio(1);
        read(0);
#pragma unroll
        for (int step = 0; step < 3 * TM; ++step) {
            const int tm = step / 3;
            if (step + 1 < 3 * TM) read(step + 1);
            if (step % 3 == 0)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn) blk[tm & 1][tn] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn)
                    blk[tm & 1][tn] =
                        __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[step & 1][h], b[tn][h], blk[tm & 1][tn], 0, 0, 0);
            if (step % 3 == 0 && tm > 0) {
                scale(tm - 1);
                // the FMAs between the MFMAs, not behind them
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);
#pragma unroll
                for (int i = 0; i < 6; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                }
                __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
        scale(TM - 1);
        wait_loads<0>();
        lds_barrier();
        cur = IMAGE - cur;
    }

    // D layout of 16x16x32: lane holds rows 4q + r, column li
    const int64_t n0 = nw + wave * 64;
    if (partial) {
        float *P = partial + (int64_t)blockIdx.z * G.n * G.rows;
        if (m0 + BM <= G.n && nw + XBN <= G.rows && G.rows * BM < (int64_t(1) << 30)) {
            // all in bounds (a uniform test), 32-bit byte offsets
            float *Pt = P + m0 * G.rows + nw;
            const uint32_t ld = (uint32_t)G.rows, c0 = (uint32_t)(wave * 64 + li);
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
    // The tile's wide rows, a bit each: two loads by the wave (a load per row
    // and store, and one row after another below, were 5 us of a call).
    uint64_t wide[2] = {};
#pragma unroll
    for (int i = 0; i < (BM + 63) / 64; ++i) {
        const int mi = 64 * i + lane;
        wide[i] = __ballot(mi < BM && m0 + mi < G.n && wflags[m0 + mi] != 0);
    }
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int mi = tm * 16 + 4 * q + r;
            const int64_t m = m0 + mi;
            if (m >= G.n || (wide[tm / 4] >> (mi & 63) & 1)) continue;
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) {
                const int64_t j = n0 + tn * 16 + li;
                if (j >= G.rows) continue;
                float v = acc[tm][tn][r];
                if (G.residual) v = G.residual[m * G.y_stride + j] + v;
                G.y[m * G.y_stride + j] = v;
            }
        }
    // this workgroup saw all of K: it recomputes its wide rows itself
    for (int i = 0; i < 2; ++i)
        for (uint64_t left = wide[i]; left; left &= left - 1) {
            const int64_t m = m0 + 64 * i + __builtin_ctzll(left), j = nw + tid;
            if (j < G.rows) G.y[m * G.y_stride + j] = wide_output(G, m, j);
        }
}

template <int FMT, int TM, int NW>
void launch_tile(hipStream_t s, const GemmArgs &a, const uint8_t *planes, float *partial, const int32_t *wflags,
                 int slices, int kper) {
    const dim3 grid((unsigned)((a.rows + 64 * NW - 1) / (64 * NW)), (unsigned)((a.n + 16 * TM - 1) / (16 * TM)),
                    (unsigned)slices);
    gemm_tall_kernel<FMT, TM, NW><<<grid, 64 * NW, 0, s>>>(a, planes, partial, wflags, kper);
}

template <int FMT>
void launch_plan(hipStream_t s, const GemmArgs &a, const TallPlan &p, const uint8_t *planes, float *partial,
                 const int32_t *wflags, int slices, int kper) {
    if (p.nw == 4) return launch_tile<FMT, 4, 4>(s, a, planes, partial, wflags, slices, kper);
    switch (p.tm) {
        case 4: return launch_tile<FMT, 4, 8>(s, a, planes, partial, wflags, slices, kper);
        case 5: return launch_tile<FMT, 5, 8>(s, a, planes, partial, wflags, slices, kper);
        case 6: return launch_tile<FMT, 6, 8>(s, a, planes, partial, wflags, slices, kper);
        case 7: return launch_tile<FMT, 7, 8>(s, a, planes, partial, wflags, slices, kper);
        default: return launch_tile<FMT, 8, 8>(s, a, planes, partial, wflags, slices, kper);
    }
}

}  // namespace

// The tile that ends first: rounds of workgroups over the 256 CUs (one of
// eight waves or two of four waves each) times a block's measured time,
// 1.3 us + 0.34 us per 16-row tile (28672 x 4096 and 6144 x 4096 Q4 at 256
// rows: 2.65 us at four tiles, 4.06 at eight; four waves 2.5).
TallPlan tall_plan(int32_t n, int64_t rows, int slices) {
    TallPlan best{8, 8};
    double cost = 1e30;
    auto consider = [&](int tm, int nw, double block) {
        const int64_t wgs = (rows + 64 * nw - 1) / (64 * nw) * ((n + 16 * tm - 1) / (16 * tm)) * slices;
        const int64_t slots = nw == 8 ? 256 : 512;
        const double c = (double)((wgs + slots - 1) / slots) * block;
        if (c < cost) {
            cost = c;
            best = TallPlan{tm, nw};
        }
    };
    consider(4, 4, 2.5);
    for (int tm = 4; tm <= 8; ++tm) consider(tm, 8, 1.3 + 0.34 * tm);
    return best;
}

size_t tall_plane_bytes(const TallPlan &p, int32_t n, int64_t cols) {
    const int64_t bm = 16 * p.tm;
    return (size_t)((n + bm - 1) / bm * bm) * (size_t)cols * 6;
}

int launch_gemm_tall(hipStream_t s, const GemmArgs &a, const TallPlan &p, uint8_t *planes, float *partial,
                     int32_t *wflags, int slices, int kper) {
    gemm_split_kernel<<<(unsigned)a.n, kSplitThreads, 0, s>>>(a.x, a.cols, a.n, 16 * p.tm, slices, planes, wflags);
    SRQ_HIP(hipGetLastError());
    if (a.fmt == SRQ_Q8)
        launch_plan<SRQ_Q8>(s, a, p, planes, partial, wflags, slices, kper);
    else
        launch_plan<SRQ_Q4>(s, a, p, planes, partial, wflags, slices, kper);
    SRQ_HIP(hipGetLastError());
    return SRQ_OK;
}

}  // namespace srq
