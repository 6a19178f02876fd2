// Q8 / Q4 weights read as whole 128-byte row segments, calls of up to 32 rows.
//
// gemm_x3_kernel loads each lane's MFMA operand straight from memory: one
// wave instruction reads 16 bytes for each of 16 feature rows x 4 K
// quarters, i.e. one 64-byte block of 16 rows, half of each of 16 cache
// lines.  Streamed alone, that pattern moves 16384 x 3072 int8 in 15.0 us
// against 9.3 us for an instruction reading 4 rows x 256 bytes (loads-only
// kernel, 256 workgroups of 8 waves, 8 loads in flight per lane): the
// memory path is bound by cache lines per instruction, not bytes.  Here a
// wave reads a pair of blocks (two 64-input blocks, 128 bytes of a row) of
// its 16 feature rows as two instructions of 8 rows x 128 bytes, stages
// them in its own LDS region and reads each block back in the operand
// layout.  A Q8 slice starting or ending on an odd block loads that block
// alone, the old way.  Q4 segments hold four blocks, counted from the slice's
// first (a slice may start inside a cache line, whose two halves are then
// two requests: still half of one per block).  Operands, MFMA order and the
// scale chain are those of gemm_x3_kernel, so every output has the same bits.
//
// A slice of more blocks than are unrolled (KU) runs in chunks of KU, each
// with its own first loads.  Measured at 32 rows, gemm_x3_kernel -> here: Q8
// 28672 x 4096 (32 blocks) 54 -> 43 us, 128256 x 3072 (48) 150 -> 128 us; Q4
// 28672 x 4096 54 -> 42 us, 6144 x 4096 (13) 19.6 -> 17.4 us, 512 x 512 (4)
// 9.6 -> 8.4 us.  What bounds it: the per-block work of a wave (code
// conversion, the activation split, LDS) at 3-4 TB/s of weights.
#include <climits>
#include <utility>

#include "gemm_x3.h"

namespace srq {
namespace {

// Region layout per 16-row tile: row r (0..15) holds its eight 16-byte
// chunks at slots chunk ^ (r % 8) ^ (r / 8), so that both the stores (8
// lanes per row) and the operand reads (16 rows per K quarter) touch
// distinct banks.
template <int FMT, int KU, int ODD>
struct PairRole {
    // Q8, block k of a slice of KU blocks whose first block has the parity
    // ODD: first(k) loads blocks k and k + 1, single(k) loads block k alone.
    // Q4: first(k) loads blocks k .. k + 3.
    static constexpr bool first(int k) { return FMT == SRQ_Q4 ? k % 4 == 0 : (k + ODD) % 2 == 0 && k + 1 < KU; }
    static constexpr bool single(int k) {
        return FMT == SRQ_Q4 ? false : (k + ODD) % 2 == 0 ? k + 1 == KU : k == 0;
    }
    static constexpr int part(int k) { return FMT == SRQ_Q4 ? k % 4 : first(k) ? 0 : 1; }
};

// f(integral_constant<int, i>) for i = 0, 1, ... in order, as straight-line code.
template <typename F, int... I>
__device__ __forceinline__ void unroll_each(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}

template <int FMT, int TM, int TN, int NW, int KU, int ODD>
__device__ __forceinline__ void x3p_slice(const GemmArgs &G, const int64_t n0, const int64_t m0, const int gbeg,
                                          const int gend, const int tid, __bf16 (*As)[3 * XTile<TM>::PLANE],
                                          u32x4v *ws, float *ss, floatx4 (&acc)[TM][TN], float &amax) {
    typedef PairRole<FMT, KU, ODD> Role;
    typedef typename XRaw<FMT>::type R;
    typedef XTile<TM, 64 * NW> X;
    constexpr int NV = X::NV, PLANE = X::PLANE, FPT = X::FPT, TPR = X::TPR;
    // Activations run one block further ahead than weights and each
    // block issues them first (Q4, whose segments are four blocks, loads
    // weights two segments ahead).  The wave's load counter retires in issue
    // order, so a wait for block k+1's activations then never waits for
    // weights issued since, and the weight loads keep DIST blocks in flight.
    constexpr int DIST = FMT == SRQ_Q4 ? 8 : 4, DA = 5;
    const int lane = tid & 63, li = lane & 15, q = lane >> 4;
    constexpr uint32_t BB = FMT == SRQ_Q8 ? kBlock : kBlock / 2;  // weight bytes per row and block
    const int64_t cols = G.cols, groups = cols / kBlock;
    const uint32_t rowb = (uint32_t)groups * BB;
    const int glast = gend - 1;
    // 32-bit offsets from the matrix base (rows * cols < 2^32): one
    // register per address instead of two
    const uint8_t *__restrict__ W = (const uint8_t *)G.values;
    uint32_t wo[TN], po[TN][2];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
        const int64_t row = n0 + tn * 16 + li;
        const int64_t rc = row < G.rows ? row : G.rows - 1;
        wo[tn] = (uint32_t)rc * rowb + 16 * q;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int64_t prow = n0 + tn * 16 + 8 * i + (lane >> 3);
            const int64_t prc = prow < G.rows ? prow : G.rows - 1;
            po[tn][i] = (uint32_t)prc * rowb;
        }
    }
    // region slots: stores of row 8i + lane/8, chunk lane%8; operand reads of row li
    const int wslot[2] = {(lane >> 3) * 8 + ((lane & 7) ^ (lane >> 3)), 64 + (lane >> 3) * 8 + ((lane & 7) ^ (lane >> 3) ^ 1)};
    const int rsw = (li & 7) ^ (li >> 3);
    const int64_t am = min(m0 + tid / TPR, (int64_t)G.n - 1);
    const float *ap = G.x + am * cols + (tid % TPR) * FPT;

    u32x4v praw[KU][TN][2], sraw[KU][TN];
    float4 areg[DA][NV];
    // The slice's scales of the workgroup's rows, loaded once in row order
    // (KU consecutive floats per row, the lanes of an instruction spanning
    // a few rows) into ss[row][block] (row stride KS, odd: the 16 rows of
    // an operand read hit distinct banks).  Per-block scale loads of 16
    // rows each would cost as many cache-line requests as the weights.
    constexpr int NT = 64 * NW, XBN = 16 * TN * NW, KS = KU | 1, SE = (XBN * KU + NT - 1) / NT;
    const int64_t wrow0 = n0 - (tid >> 6) * 16 * TN;  // the workgroup's first output
    float sreg[SE];
#pragma unroll
    for (int i = 0; i < SE; ++i) {
        const int e = tid + NT * i;
        const int r = e / KU, j = e - r * KU;
        const int64_t row = min(wrow0 + r, G.rows - 1);
        // a block past the slice's end (last slice) is added with a zero scale
        sreg[i] = e < XBN * KU && gbeg + j < gend ? G.scales[row * groups + min(gbeg + j, glast)] : 0.0f;
    }
    auto stage_s = [&]() {
#pragma unroll
        for (int i = 0; i < SE; ++i) {
            const int e = tid + NT * i;
            const int r = e / KU, j = e - r * KU;
            if (e < XBN * KU) ss[r * KS + j] = sreg[i];
        }
    };
    const float *sl = ss + ((tid >> 6) * 16 * TN + li) * KS;  // this lane's rows
    // Weight loads of block j (its scale, and its pair or its lone block).
    // A phantom block past the slice's end (last slice) reads clamped,
    // in-row data and is added with a zero scale.
    auto load_w = [&](auto J) {
        constexpr int j = decltype(J)::value;
        if constexpr (j < KU) {
            const int g = gbeg + j;
            if constexpr (Role::first(j)) {
                // Q8 pairs are aligned, so only a phantom one is clamped; of
                // a Q4 segment the chunks past the row's end are.
                const uint32_t pg = FMT == SRQ_Q8
                                        ? (uint32_t)min((int64_t)g, groups - 2) * BB + 16 * (lane & 7)
                                        : min((uint32_t)g * BB + 16 * (lane & 7), rowb - 16);
#pragma unroll
                for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                    for (int i = 0; i < 2; ++i) praw[j][tn][i] = *(const u32x4v *)(W + (uint64_t)(po[tn][i] + pg));
            } else if constexpr (Role::single(j)) {
                const uint32_t sg = (uint32_t)min(g, glast) * BB;
#pragma unroll
                for (int tn = 0; tn < TN; ++tn) sraw[j][tn] = *(const u32x4v *)(W + (uint64_t)(wo[tn] + sg));
            }
        }
    };
    auto load_a = [&](auto J) {
        constexpr int j = decltype(J)::value;
        if constexpr (j < KU) {
            const int64_t g = min(gbeg + j, glast);
#pragma unroll
            for (int i = 0; i < NV; ++i) areg[j % DA][i] = *(const float4 *)(ap + g * kBlock + 4 * i);
        }
    };
    auto stage_w = [&](auto J) {
        constexpr int j = decltype(J)::value;
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
            for (int i = 0; i < 2; ++i) ws[tn * 128 + wslot[i]] = praw[j][tn][i];
    };

    // issue order A0, A1, W0, A2, W1, ..., A(DA-1), W(DIST-1): each
    // block's weights after the activations one block further on
    load_a(std::integral_constant<int, 0>{});
    unroll_each([&](auto J) {
        constexpr int j = decltype(J)::value;
        if constexpr (j + 1 < DA) load_a(std::integral_constant<int, j + 1>{});
        load_w(J);
    }, std::make_integer_sequence<int, DIST>{});
    stage_s();
    if constexpr (Role::first(0)) stage_w(std::integral_constant<int, 0>{});
    amax = fmaxf(amax, xstore_a<TM, NT>(As[0], tid, areg[0]));
    lds_barrier();

    unroll_each([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int u = k & 1, v = u ^ 1;
        bf16x8 b[TN][2];
        if constexpr (Role::single(k)) {
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) xcodes<SRQ_Q8>(sraw[k][tn], b[tn][0], b[tn][1]);
        } else if constexpr (FMT == SRQ_Q8) {
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
                xcodes<SRQ_Q8>(ws[tn * 128 + li * 8 + ((4 * Role::part(k) + q) ^ rsw)], b[tn][0], b[tn][1]);
        } else {
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
                xcodes<SRQ_Q4>(((const R *)&ws[tn * 128 + li * 8 + ((2 * Role::part(k) + (q >> 1)) ^ rsw)])[q & 1],
                               b[tn][0], b[tn][1]);
        }
        __builtin_amdgcn_sched_barrier(0);
        load_a(std::integral_constant<int, k + DA>{});
        load_w(std::integral_constant<int, k + DIST>{});
        __builtin_amdgcn_sched_barrier(0);
        const __bf16 *as = As[u];
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            bf16x8 a[3][2];
#pragma unroll
            for (int t = 0; t < 3; ++t)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    a[t][h] = *(const bf16x8 *)(as + t * PLANE + (tm * 16 + li) * XLD + 16 * q + 8 * h);
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) {
                floatx4 blk = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int t = 2; t >= 0; --t)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        blk = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t][h], b[tn][h], blk, 0, 0, 0);
                const float sc_u = FMT == SRQ_Q4 ? 16.0f * sl[tn * 16 * KS + k] : sl[tn * 16 * KS + k];
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[tm][tn][r] = __builtin_fmaf(blk[r], sc_u, acc[tm][tn][r]);
            }
        }
        if constexpr (k + 1 < KU) {
            // the next pair -> the region (after this block's reads of it),
            // block k+1's activations -> the other stage
            if constexpr (Role::first(k + 1)) stage_w(std::integral_constant<int, k + 1>{});
            amax = fmaxf(amax, xstore_a<TM, NT>(As[v], tid, areg[(k + 1) % DA]));
            lds_barrier();
        }
    }, std::make_integer_sequence<int, KU>{});
}

// 16- or 32-row tiles, cols % 128 == 0 (Q8) or cols % 64 == 0 (Q4), rows * cols
// < 2^32.  Slices of KU blocks, or (MULTI) of several chunks of KU; the last
// slice and the last chunk may be shorter.  NW waves of TN feature tiles each.
// Eight waves keep two per SIMD in the one workgroup a CU holds, so that
// one wave's MFMAs overlap another's conversions and LDS waits, while the
// activation stage stays shared by all the workgroup's features.  Up to
// eight tiles per workgroup, two workgroups fit a CU.
template <int FMT, int TM, int TN, int NW, int KU, bool MULTI>
__global__ __launch_bounds__(64 * NW, TN * NW <= 8 ? 2 : 1) void gemm_x3p_kernel(
    const GemmArgs G, float *__restrict__ partial, int32_t *__restrict__ wflags, const int kper) {
    constexpr int BM = XTile<TM>::BM, PLANE = XTile<TM>::PLANE, XBN = 16 * TN * NW;
    __shared__ __attribute__((aligned(16))) __bf16 As[2][3 * PLANE];
    __shared__ u32x4v Ws[NW][TN * 128];
    __shared__ float Ss[XBN * (KU | 1)];
    __shared__ int row_wide[BM];
    const int tid = threadIdx.x, wave = tid >> 6;
    const int64_t n0 = (int64_t)blockIdx.x * XBN + wave * 16 * TN, m0 = (int64_t)blockIdx.y * BM;
    const int groups = (int)(G.cols / kBlock);
    const int gbeg = (int)blockIdx.z * kper;
    const int gend = min(gbeg + kper, groups);
    if (tid < BM) row_wide[tid] = 0;
    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    float amax = 0.0f;
    auto chunk = [&](const int c, const int end) {
        if (FMT == SRQ_Q8 && (c & 1))
            x3p_slice<FMT, TM, TN, NW, KU, 1>(G, n0, m0, c, end, tid, As, Ws[wave], Ss, acc, amax);
        else
            x3p_slice<FMT, TM, TN, NW, KU, 0>(G, n0, m0, c, end, tid, As, Ws[wave], Ss, acc, amax);
    };
    if constexpr (MULTI) {
        for (int c = gbeg; c < gend; c += KU) {
            chunk(c, min(c + KU, gend));
            lds_barrier();  // the stages and scales are read before the next chunk's
        }
    } else {
        chunk(gbeg, gend);
    }
    x3_finish<TM, TN, XBN, 64 * NW>(G, partial, wflags, acc, amax, row_wide, n0, m0, tid);
}

struct PairCall {
    hipStream_t s;
    dim3 grid;
    const GemmArgs &a;
    float *partial;
    int32_t *wflags;
    int kper;
};

template <int FMT, int TM, int TN, int NW, int KU, bool MULTI>
void launch(const PairCall &c) {
    gemm_x3p_kernel<FMT, TM, TN, NW, KU, MULTI><<<c.grid, 64 * NW, 0, c.s>>>(c.a, c.partial, c.wflags, c.kper);
}

// Slices of 4..16 blocks: the kernel unrolled over exactly them.
template <int FMT, int TM, int TN, int NW, int KU = 4>
void launch_exact(const PairCall &c) {
    if constexpr (KU <= 16) {
        if (c.kper == KU)
            launch<FMT, TM, TN, NW, KU, false>(c);
        else
            launch_exact<FMT, TM, TN, NW, KU + 1>(c);
    }
}

// Blocks per chunk of a slice of kper > 16 blocks: the cheapest, counting the
// blocks of a short last chunk (it runs them all) and two for each chunk's
// first loads.  Nine and ten are there for slices just past 16 blocks: in
// chunks of 12, 17 or 18 blocks ran 24 (8192 features in four slices, 24 rows,
// Q4: 17 / 18 / 19 blocks 25.3 -> 21.4 / 21.4 / 22.5 us; gemm_x3_kernel 22.0 /
// 23.1 / 24.0).  Eleven, 13 and 15 would gain up to 6% at 21, 26 and 30 blocks
// for 48 more kernels.
int chunk_blocks(int kper) {
    int best = 0, cost = INT_MAX;
    for (const int ku : {16, 14, 12, 10, 9}) {
        const int c = (kper + ku - 1) / ku * (ku + 2);
        if (c < cost) cost = c, best = ku;
    }
    return best;
}

template <int FMT, int TM, int TN, int NW>
void launch_chunks(const PairCall &c) {
    switch (chunk_blocks(c.kper)) {
        case 16: return launch<FMT, TM, TN, NW, 16, true>(c);
        case 14: return launch<FMT, TM, TN, NW, 14, true>(c);
        case 12: return launch<FMT, TM, TN, NW, 12, true>(c);
        case 10: return launch<FMT, TM, TN, NW, 10, true>(c);
        default: return launch<FMT, TM, TN, NW, 9, true>(c);
    }
}

template <int FMT, int TM, int TN, int NW>
void launch_pairs(const PairCall &c) {
    c.kper <= 16 ? launch_exact<FMT, TM, TN, NW>(c) : launch_chunks<FMT, TM, TN, NW>(c);
}

template <int FMT>
void launch_fmt(const PairCall &c, int bm, int tn) {
    // the plan's feature tile (64 * tn); 256 features at 32 rows over 8 waves
    // (gate/up 16384x3072 Q8 at 17-32 rows: 24.5 -> 22.6 us; 128 features
    // over 8 waves were slower, and so were 128 over 4 for slices run in
    // chunks: 32768x4096 44 -> 47 us)
    if (bm == 32)
        tn == 2 ? launch_pairs<FMT, 2, 2, 4>(c) : launch_pairs<FMT, 2, 2, 8>(c);
    else
        tn == 1 ? launch_pairs<FMT, 1, 1, 4>(c) : launch_pairs<FMT, 1, 2, 4>(c);
}

}  // namespace

bool gemm_pairs_ok(const GemmArgs &a, int kper) {
    if ((uint64_t)a.rows * (uint64_t)a.cols > UINT32_MAX || kper < 4) return false;
    return a.fmt == SRQ_Q8 ? a.cols % (2 * kBlock) == 0 : a.fmt == SRQ_Q4 && a.cols % kBlock == 0;
}

void launch_gemm_pairs(hipStream_t s, const GemmArgs &a, int bm, int tn, float *partial, int32_t *wflags, int slices,
                       int kper) {
    const int xbn = 64 * tn;
    const dim3 grid((unsigned)((a.rows + xbn - 1) / xbn), (unsigned)((a.n + bm - 1) / bm), (unsigned)slices);
    const PairCall c{s, grid, a, partial, wflags, kper};
    a.fmt == SRQ_Q8 ? launch_fmt<SRQ_Q8>(c, bm, tn) : launch_fmt<SRQ_Q4>(c, bm, tn);
}

}  // namespace srq
