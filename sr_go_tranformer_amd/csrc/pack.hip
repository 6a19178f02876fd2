// On-device Q8/Q4 packing and dequantization for gfx950.
//
// Packing restates the reference's streaming packer bit for bit
// (cmd/monolith/monolith.go: readParam M:857-880, lowBitScale M:3877-3891,
// q8Value M:3893-3898, putQuantized M:3840-3850, q4 put M:3819-3822,
// source decode M:884-920, halfFloat M:838-850).  Eight lanes own one
// 64-column block of one row, eight consecutive columns each; the block amax
// is a maximum over the eight lanes (exact in any order).
#include <type_traits>

#include "srq_internal.h"

namespace srq {
namespace {

// halfFloat (M:838-850): exact, including signed zero and subnormals.
__device__ inline float half_bits_to_float(uint32_t v) {
    uint32_t sign = (v & 0x8000u) << 16;
    uint32_t exp = (v >> 10) & 31u, frac = v & 1023u;
    if (exp == 0) {
        float x = (float)frac * 0x1p-24f;  // exact: frac < 2^10
        return __uint_as_float(__float_as_uint(x) | sign);
    }
    if (exp == 31) return __uint_as_float(sign | 0x7f800000u | (frac << 13));
    return __uint_as_float(sign | ((exp + 112u) << 23) | (frac << 13));
}

__device__ inline float load_src(const void *src, int64_t i, int dtype) {
    if (dtype == SRQ_SRC_F32) return ((const float *)src)[i];
    uint32_t w = ((const uint16_t *)src)[i];
    if (dtype == SRQ_SRC_BF16) return __uint_as_float(w << 16);
    return half_bits_to_float(w);
}

// lowBitScale (M:3877-3891).
__device__ inline float low_bit_scale(float amax, double levels) {
    if (amax == 0.0f) return 0.0f;
    float scale = (float)((double)amax / levels);
    const float tiny = __uint_as_float(1u);
    if (scale == 0.0f) return tiny;
    if (scale > tiny && (double)scale * levels > (double)amax) scale = __uint_as_float(__float_as_uint(scale) - 1u);
    return scale;
}

// q8Value / putQuantized: clamp(round_half_away(f64(v)/f64(scale))).
__device__ inline int quant_code(float v, float scale, double lim) {
    if (scale == 0.0f) return 0;
    double q = round((double)v / (double)scale);
    q = q > lim ? lim : q;
    q = q < -lim ? -lim : q;
    return (int)q;
}

// Largest value of the eight lanes that share a block (lane ^ 1, ^ 2, then
// the other quad of the half row).
__device__ __forceinline__ uint32_t max8(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true));   // quad_perm [2,3,0,1]
    return max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, true));  // row_half_mirror
}

// The block's scale and its lane's eight codes, with the results of
// low_bit_scale and quant_code.  Those divide in FP64, which bounded the
// packer: about 30 double-rate instructions per element, 235 us for a
// 14336 x 4096 bf16 source (0.8 TB/s).  For scales in the normal range the
// same values come from FP32:
//  - scale: amax / 127 (or 7) lies no nearer to the midpoint of two floats
//    than 2^-32 of its value (127 and 7 are odd, so a midpoint times either
//    needs more bits than amax has), so rounding the FP64 quotient to FP32 gives the
//    FP32 quotient; the overshoot test is the sign of one exact-product FMA.
//  - code: k = rint(v * rcp(scale)) is off by at most one, and only when
//    v / scale is within 2^-15 of a half integer.  r = v - k * scale then
//    decides; unless some |r| of the lane is within 2^-13 of scale / 2
//    (FP32 rounding of r is 2^-23 of it), k is the rounded quotient.
//    Otherwise r is formed exactly, in FP64 (k * scale has 32 bits), and
//    compared with scale / 2, a tie going away from zero; v / scale is no
//    nearer to a half integer than 2^-26 unless it is one, so rounding the
//    FP64 quotient gives the same code.  (bf16 blocks hold exact ties in
//    numbers: dividing there, a call below took 73 us instead of 57.)
// amax: bits of the block's largest |v| (a NaN's are above an infinity's).
template <int FMT>
__device__ __forceinline__ float quant8(const float (&v)[8], uint32_t amax_bits, int (&code)[8]) {
    constexpr float L = FMT == SRQ_Q8 ? 127.0f : 7.0f;
    const float amax = __uint_as_float(amax_bits);
    if (amax > 0x1p-90f && amax < 0x1p120f) {
        float scale = __fdiv_rn(amax, L);
        if (__builtin_fmaf(scale, L, -amax) > 0.0f) scale = __uint_as_float(__float_as_uint(scale) - 1u);
        const float inv = __builtin_amdgcn_rcpf(scale);
        float far = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float k = __builtin_rintf(v[j] * inv);
            far = fmaxf(far, fabsf(__builtin_fmaf(-k, scale, v[j])));
            code[j] = (int)k;
        }
        if (far > scale * (0.5f - 0x1p-14f)) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const double r = __builtin_fma(-(double)code[j], (double)scale, (double)v[j]), h = 0.5 * (double)scale;
                const bool neg = v[j] < 0.0f;
                code[j] += (neg ? r > h : r >= h) ? 1 : (neg ? r <= -h : r < -h) ? -1 : 0;
            }
        }
        return scale;
    }
    // zero, tiny, huge and non-finite blocks
    const float top = amax_bits > 0x7f800000u ? __uint_as_float(0x7f800000u) : amax;
    const float scale = low_bit_scale(top, (double)L);
#pragma unroll
    for (int j = 0; j < 8; ++j) code[j] = quant_code(v[j], scale, (double)L);
    return scale;
}

template <int DT>
__device__ __forceinline__ float decode_src(uint32_t bits) {
    if constexpr (DT == SRQ_SRC_F32) return __uint_as_float(bits);
    if constexpr (DT == SRQ_SRC_BF16) return __uint_as_float(bits << 16);
    return half_bits_to_float(bits);
}

constexpr int kPackBlocks = 32;  // blocks per 256-thread workgroup

// VEC: cols % 64 == 0 and 16-byte aligned sources: a matrix is then one run
// of whole blocks, and a lane reads its eight columns as one (bf16, f16) or
// two (f32) 16-byte loads and writes one 8-byte (Q8) or 4-byte (Q4) word.
// Bound by HBM.  Otherwise (odd
// widths, unaligned pointers) the same eight columns go one at a time.
// One lane per element and FP64 divisions before; 14336 x 4096 to Q8, kernel
// alone: bf16 235 -> 43 us (4.2 TB/s), f32 51 us (5.8 TB/s); whole calls at
// width 4095: bf16 to Q8 257 -> 96 us, f32 to Q4 273 -> 119 us.  Two or four
// blocks per lane measured no faster (4095 wide: 122-128 us).
template <int FMT, int DT, bool VEC>
__global__ __launch_bounds__(256) void pack_kernel(const int64_t rows, const int64_t cols,
                                                   const void *__restrict__ src, void *__restrict__ values,
                                                   float *__restrict__ scales, int *__restrict__ err_flag) {
    const int sub = threadIdx.x & 7;
    const int64_t groups = groups_of(cols);
    const int64_t b = (int64_t)blockIdx.x * kPackBlocks + (threadIdx.x >> 3);
    if (b >= rows * groups) return;  // the eight lanes of a block agree
    const int64_t row = VEC ? 0 : b / groups;
    const int64_t col = VEC ? 0 : (b - row * groups) * kBlock + 8 * sub;  // the lane's first column
    const int64_t at = VEC ? b * kBlock + 8 * sub : row * cols + col;
    uint32_t raw[8] = {};
    if constexpr (VEC && DT == SRQ_SRC_F32) {
        const uint4 p = ld_stream16((const uint32_t *)src + at), q = ld_stream16((const uint32_t *)src + at + 4);
        raw[0] = p.x, raw[1] = p.y, raw[2] = p.z, raw[3] = p.w;
        raw[4] = q.x, raw[5] = q.y, raw[6] = q.z, raw[7] = q.w;
    } else if constexpr (VEC) {
        const uint4 p = ld_stream16((const uint16_t *)src + at);
        const uint32_t w[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) raw[2 * j] = w[j] & 0xFFFFu, raw[2 * j + 1] = w[j] >> 16;
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (col + j < cols)
                raw[j] = DT == SRQ_SRC_F32 ? ((const uint32_t *)src)[at + j] : ((const uint16_t *)src)[at + j];
    }
    float v[8];
    uint32_t amax = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        v[j] = decode_src<DT>(raw[j]);
        amax = max(amax, __float_as_uint(v[j]) & 0x7fffffffu);
    }
    amax = max8(amax);
    if (amax >= 0x7f800000u) err_flag[0] = 1;
    int code[8];
    const float scale = quant8<FMT>(v, amax, code);
    if (sub == 0) scales[b] = scale;
    if constexpr (VEC && FMT == SRQ_Q8) {
        uint32_t w[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
            w[i] = ((uint32_t)code[4 * i] & 255u) | ((uint32_t)code[4 * i + 1] & 255u) << 8 |
                   ((uint32_t)code[4 * i + 2] & 255u) << 16 | (uint32_t)code[4 * i + 3] << 24;
        *(uint2 *)((uint8_t *)values + at) = make_uint2(w[0], w[1]);
    } else if constexpr (VEC) {
        uint32_t w = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) w |= ((uint32_t)code[j] & 15u) << (4 * j);
        *(uint32_t *)((uint8_t *)values + at / 2) = w;
    } else if constexpr (FMT == SRQ_Q8) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (col + j < cols) ((int8_t *)values)[at + j] = (int8_t)code[j];
    } else {
        // Low nibble = even column, high nibble = odd column; an odd row
        // width leaves a zero high pad nibble (M:3819-3822): a column past
        // the end was read as zero.
        uint8_t *out = (uint8_t *)values + row * ((cols + 1) / 2) + col / 2;
#pragma unroll
        for (int j = 0; j < 8; j += 2)
            if (col + j < cols) out[j / 2] = (uint8_t)(((uint32_t)code[j] & 15u) | ((uint32_t)code[j + 1] & 15u) << 4);
    }
}

__global__ __launch_bounds__(256) void convert_kernel(int64_t count, const void *__restrict__ src, int dtype,
                                                      float *__restrict__ dst, int *__restrict__ err_flag) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count; i += (int64_t)gridDim.x * 256) {
        float v = load_src(src, i, dtype);
        if (!isfinite(v)) err_flag[0] = 1;
        dst[i] = v;
    }
}

// copyRow (M:3900-3921): dst = f32(code) * scale, one rounding.
template <int FMT>
__global__ __launch_bounds__(256) void dequant_kernel(int64_t cols, const void *__restrict__ values,
                                                      const float *__restrict__ scales,
                                                      const int32_t *__restrict__ rows, float *__restrict__ dst) {
    const int64_t groups = groups_of(cols);
    const int64_t r = rows[blockIdx.y];
    float *out = dst + (int64_t)blockIdx.y * cols;
    for (int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x; j < cols; j += (int64_t)gridDim.x * 256) {
        float w;
        if (FMT == SRQ_F32) {
            out[j] = ((const float *)values)[r * cols + j];
            continue;
        } else if (FMT == SRQ_Q8) {
            w = (float)((const int8_t *)values)[r * cols + j];
        } else {
            uint32_t b = ((const uint8_t *)values)[r * ((cols + 1) / 2) + j / 2];
            uint32_t nib = (j & 1) ? (b >> 4) : (b & 15u);
            w = (float)(((int32_t)(nib << 28)) >> 28);
        }
        out[j] = w * scales[r * groups + j / kBlock];
    }
}

// SplitMix64 output number k (k >= 1) from state `seed` (M:1416-1422):
// the state after k calls is seed + k*gamma, so draws are independent.
__device__ inline uint64_t splitmix_at(uint64_t seed, uint64_t k) {
    uint64_t z = seed + k * 0x9e3779b97f4a7c15ULL;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
    return z ^ (z >> 31);
}

// dst[i] = f32(Normal() * scale) where Normal uses draws 2i+1 and 2i+2
// (RNG.Normal M:1437-1439, random init M:5218).
__global__ __launch_bounds__(256) void fill_normal_kernel(float *__restrict__ dst, int64_t count, uint64_t seed,
                                                          double scale) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count; i += (int64_t)gridDim.x * 256) {
        const double u1 = (double)(splitmix_at(seed, 2 * (uint64_t)i + 1) >> 11) * (1.0 / 9007199254740992.0);
        const double u2 = (double)(splitmix_at(seed, 2 * (uint64_t)i + 2) >> 11) * (1.0 / 9007199254740992.0);
        const double nrm = sqrt(-2.0 * log(1.0 - u1)) * cos(2.0 * M_PI * u2);
        dst[i] = (float)(nrm * scale);
    }
}

}  // namespace

int launch_fill_normal(hipStream_t s, float *dst, int64_t count, uint64_t seed, double scale) {
    if (count <= 0) return SRQ_OK;
    int64_t blocks = (count + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    fill_normal_kernel<<<(unsigned)blocks, 256, 0, s>>>(dst, count, seed, scale);
    SRQ_HIP(hipGetLastError());
    return SRQ_OK;
}

template <int FMT, int DT>
void launch_pack_as(hipStream_t s, int64_t rows, int64_t cols, const void *src, void *values, float *scales,
                    int *err_flag) {
    const dim3 grid((unsigned)((rows * groups_of(cols) + kPackBlocks - 1) / kPackBlocks));
    if (cols % kBlock == 0 && ((uintptr_t)src & 15) == 0 && ((uintptr_t)values & 7) == 0)
        pack_kernel<FMT, DT, true><<<grid, 256, 0, s>>>(rows, cols, src, values, scales, err_flag);
    else
        pack_kernel<FMT, DT, false><<<grid, 256, 0, s>>>(rows, cols, src, values, scales, err_flag);
}

int launch_pack(hipStream_t s, int fmt, int64_t rows, int64_t cols, const void *src, int dtype, void *values,
                float *scales, int *err_flag) {
    if (rows <= 0 || cols <= 0) return SRQ_OK;
    auto go = [&](auto F) {
        constexpr int FMT = decltype(F)::value;
        if (dtype == SRQ_SRC_F32)
            launch_pack_as<FMT, SRQ_SRC_F32>(s, rows, cols, src, values, scales, err_flag);
        else if (dtype == SRQ_SRC_BF16)
            launch_pack_as<FMT, SRQ_SRC_BF16>(s, rows, cols, src, values, scales, err_flag);
        else
            launch_pack_as<FMT, SRQ_SRC_F16>(s, rows, cols, src, values, scales, err_flag);
    };
    if (fmt == SRQ_Q8)
        go(std::integral_constant<int, SRQ_Q8>{});
    else
        go(std::integral_constant<int, SRQ_Q4>{});
    SRQ_HIP(hipGetLastError());
    return SRQ_OK;
}

int launch_convert_f32(hipStream_t s, int64_t count, const void *src, int dtype, float *dst, int *err_flag) {
    if (count <= 0) return SRQ_OK;
    int64_t blocks = (count + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    convert_kernel<<<(unsigned)blocks, 256, 0, s>>>(count, src, dtype, dst, err_flag);
    SRQ_HIP(hipGetLastError());
    return SRQ_OK;
}

int launch_dequant_rows(hipStream_t s, int fmt, int64_t cols, const void *values, const float *scales,
                        const int32_t *rows, int32_t count, float *dst) {
    if (count <= 0 || cols <= 0) return SRQ_OK;
    int64_t bx = (cols + 255) / 256;
    if (bx > 64) bx = 64;
    dim3 grid((unsigned)bx, (unsigned)count);
    if (fmt == SRQ_Q8)
        dequant_kernel<SRQ_Q8><<<grid, 256, 0, s>>>(cols, values, scales, rows, dst);
    else if (fmt == SRQ_Q4)
        dequant_kernel<SRQ_Q4><<<grid, 256, 0, s>>>(cols, values, scales, rows, dst);
    else
        dequant_kernel<SRQ_F32><<<grid, 256, 0, s>>>(cols, values, scales, rows, dst);
    SRQ_HIP(hipGetLastError());
    return SRQ_OK;
}

}  // namespace srq
