// GEMM of F32 weights on FP32 MFMA (v_mfma_f32_16x16x4f32): linearFP32Range
// (cmd/monolith/monolith.go M:3942-4780) for prefill chunks and batched steps.
//
// F32 operands need no conversion, so both go from memory to LDS by
// LDS-direct loads, D - 1 K steps of 32 ahead: a step's MFMAs take 0.4 us (32
// rows) or 0.85 us (64 rows) on a SIMD, memory answers in 1-2 us, and one
// step of prefetch through registers left the matrix cores waiting (3072 x 576
// at 129 rows: 1.9 us a step).  Workgroup tile BM rows x 128 features, 4 waves of
// 32 rows x (128 / waves across features).  Within a K step, MFMA step s
// feeds lane group g (lane / 16) the K index 8g + s, so every lane reads its 8
// values of a row as two 16-byte reads; chunk c of row r sits at slot
// c ^ (r % 8), so that a read of one chunk of 16 rows touches every bank once.
//
// Measured, whole srq_linear call with its reduction, before -> now: 3072 x 576
// at 129 rows 21.0 -> 13.5 us, 49152 x 576 at 32 / 1024 rows 47.3 -> 36.5 / 745
// -> 532 us (109 TFLOP/s of 157), 4096 x 2048 at 256 rows 67.8 -> 52.2 us.
// What bounds it now: the FP32 MFMAs at many rows, the load latency of the
// first steps and the two launches at few.
#include "gemm_common.h"

namespace srq {
namespace {

constexpr int BN = 128, BK = 32;
constexpr int kStepBytes = BK * 4;  // one row of one step

struct __attribute__((packed, aligned(4))) Loose {  // 16 bytes at any float
    float v[4];
};

template <int BM>
struct F32Tile {
    static constexpr int STAGE = (BM + BN) * kStepBytes;
    static constexpr int LOADS = STAGE / 1024 / 4;  // per wave and step
};

// Slices, partial and wflags as gemm_kernel (gemm.hip); kper counts K steps.
// D: K steps the LDS ring holds.  DIRECT: operands 16-byte aligned, loaded
// straight to LDS.  Otherwise (D = 2) they pass through registers: step k + 1
// is in flight during the MFMAs of step k and stored after them (loaded and
// stored before them, every step waited for memory: activations off by one
// float, 49152 x 576 at 32 / 1000 rows 46 -> 29 / 724 -> 502 us, 3072 x 576 at
// 129 rows 15.8 -> 14.5 us).
template <int BM, int D, bool DIRECT>
__global__ __launch_bounds__(256, 1) void gemm_f32_kernel(const GemmArgs G, float *__restrict__ partial,
                                                          int32_t *__restrict__ wflags, const int kper) {
    typedef F32Tile<BM> T;
    constexpr int WM = BM / 32, WN = 4 / WM, TN = BN / WN / 16;
    __shared__ __attribute__((aligned(16))) uint8_t ring[D][T::STAGE];
    __shared__ int row_wide[BM];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN, gq = lane >> 4, li = lane & 15;
    const int64_t n0 = (int64_t)blockIdx.x * BN, m0 = (int64_t)blockIdx.y * BM;
    const int kbeg = (int)blockIdx.z * kper;
    const int kend = min(kbeg + kper, (int)(G.cols / BK));
    if (tid < BM) row_wide[tid] = 0;

    // A step's stage: BM activation rows, then 128 feature rows.  Load j of
    // this wave brings 8 rows x 128 bytes; rows past the ends read the last
    // row and are never stored.
    const uint8_t *src[T::LOADS];
#pragma unroll
    for (int j = 0; j < T::LOADS; ++j) {
        const int r = (j * 4 + wave) * 8 + (lane >> 3);
        const int64_t chunk = (lane & 7) ^ (r & 7);
        const float *row = r < BM ? G.x + min(m0 + r, (int64_t)G.n - 1) * G.cols
                                  : (const float *)G.values + min(n0 + r - BM, G.rows - 1) * G.cols;
        src[j] = (const uint8_t *)(row + (int64_t)kbeg * BK) + chunk * 16;
    }
    const uint32_t ring0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)&ring[0][0];
    auto step_off = [&](const int k) { return (int64_t)(min(k, kend - 1) - kbeg) * kStepBytes; };
    auto load = [&](const int k, const uint32_t slot) {
#pragma unroll
        for (int j = 0; j < T::LOADS; ++j)
            lds_load16(ring0 + slot + (uint32_t)((j * 4 + wave) * 1024), src[j] + step_off(k));
    };
    Loose held[DIRECT ? 1 : T::LOADS];
    auto fetch = [&](const int k) {
#pragma unroll
        for (int j = 0; j < T::LOADS; ++j) held[j] = *(const Loose *)(src[j] + step_off(k));
    };
    auto put = [&](const uint32_t slot) {
#pragma unroll
        for (int j = 0; j < T::LOADS; ++j)
            *(floatx4 *)(&ring[0][0] + slot + (j * 4 + wave) * 1024 + lane * 16) =
                floatx4{held[j].v[0], held[j].v[1], held[j].v[2], held[j].v[3]};
    };

    floatx4 acc[2][TN];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    float amax[2] = {0.f, 0.f};
    if constexpr (DIRECT) {
#pragma unroll
        for (int d = 0; d < D - 1; ++d) load(kbeg + d, (uint32_t)(d * T::STAGE));
    } else {
        fetch(kbeg);
        put(0);
        fetch(kbeg + 1);
    }
    // operand chunks 2gq and 2gq + 1 of row li of a tile
    const int rd[2] = {((2 * gq) ^ (li & 7)) * 16 + li * kStepBytes, ((2 * gq + 1) ^ (li & 7)) * 16 + li * kStepBytes};
    uint32_t cur = 0, fill = (D - 1) * T::STAGE;
    for (int k = kbeg; k < kend; ++k) {
        // Step k has landed when at most the D - 2 later steps' loads are
        // outstanding; past the barrier every wave's share of it has, and no
        // wave reads step k - 1, whose slot the next load fills.
        if constexpr (DIRECT) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 2) * T::LOADS) : "memory");
        lds_barrier();
        if constexpr (DIRECT) load(k + D - 1, fill);
        const uint8_t *as = &ring[0][0] + cur, *bs = as + BM * kStepBytes;
        float af[2][8], bf[TN][8];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const floatx4 v = *(const floatx4 *)(as + (wm * 32 + t * 16) * kStepBytes + rd[h]);
#pragma unroll
                for (int e = 0; e < 4; ++e) af[t][4 * h + e] = v[e];
            }
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const floatx4 v = *(const floatx4 *)(bs + (wn * TN + t) * 16 * kStepBytes + rd[h]);
#pragma unroll
                for (int e = 0; e < 4; ++e) bf[t][4 * h + e] = v[e];
            }
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int tm = 0; tm < 2; ++tm) {
#pragma unroll
                for (int tn = 0; tn < TN; ++tn)
                    acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[tm][s], bf[tn][s], acc[tm][tn], 0, 0, 0);
                amax[tm] = fmaxf(amax[tm], fabsf(af[tm][s]));
            }
        if constexpr (!DIRECT) {
            put(fill);
            fetch(k + 2);
        }
        cur = cur == (D - 1) * T::STAGE ? 0 : cur + T::STAGE;
        fill = fill == (D - 1) * T::STAGE ? 0 : fill + T::STAGE;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int t = 0; t < 2; ++t)
        if (amax[t] > kWideLimit) row_wide[wm * 32 + t * 16 + li] = 1;
    __syncthreads();
    gemm_finish<BM, BN, 2, TN>(G, partial, wflags, acc, row_wide, n0, m0, wm * 32, wn * TN * 16, tid);
}

}  // namespace

int launch_gemm_f32(hipStream_t s, const GemmArgs &a, float *partial, int32_t *wflags, int slices, int kper) {
    const int64_t ft = (a.rows + BN - 1) / BN * slices;
    // 32-row tiles, one workgroup per CU with six steps in LDS, for calls that
    // are one round of them; past that 64-row tiles, whose two workgroups
    // per CU cover each other's first loads (3072 x 576 at 256 rows, 384
    // workgroups of 32 rows: 23.4 us; 192 of 64: 20.6).  Slices of a few
    // steps load no more than they have.
    const int64_t wg32 = ft * ((a.n + 31) / 32);
    const int bm = a.n <= 32 || wg32 <= 256 ? 32 : 64;
    const dim3 grid((unsigned)((a.rows + BN - 1) / BN), (unsigned)((a.n + bm - 1) / bm), (unsigned)slices);
    const bool loose = (((uintptr_t)a.x) | ((uintptr_t)a.values)) & 15;
    if (loose && bm == 64)
        gemm_f32_kernel<64, 2, false><<<grid, 256, 0, s>>>(a, partial, wflags, kper);
    else if (loose)
        gemm_f32_kernel<32, 2, false><<<grid, 256, 0, s>>>(a, partial, wflags, kper);
    else if (bm == 64)
        gemm_f32_kernel<64, 3, true><<<grid, 256, 0, s>>>(a, partial, wflags, kper);
    else if (kper > 4)
        gemm_f32_kernel<32, 6, true><<<grid, 256, 0, s>>>(a, partial, wflags, kper);
    else
        gemm_f32_kernel<32, 3, true><<<grid, 256, 0, s>>>(a, partial, wflags, kper);
    SRQ_HIP(hipGetLastError());
    return SRQ_OK;
}

}  // namespace srq
