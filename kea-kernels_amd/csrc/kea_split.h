// FP32 operands as pairs of FP16 values for the FP16 matrix cores: x * 2^a = hi + lo with a power of two a per row (or
// group of rows) that puts the largest magnitude into [2^14, 2^15). hi + lo holds every element to 2^-22 of itself or 2^-39
// of that largest one, whatever the range of the input; a product is three FP16 MFMAs with FP32 accumulation (hi hi +
// hi lo + lo hi; the dropped lo lo term is 2^-22 of the product, of random sign). Infinities have no such scale: the
// kernels look for them and take a plain FP32 path.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kea_wave.h"

namespace kea {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

// The binary exponent e of a magnitude given by its bits (2^e <= m < 2^(e+1)), clamped so that 2^(14-e) and 2^(e-14)
// are normal numbers.
__device__ __forceinline__ int exponent_of(int bits) { return min(max((bits >> 23) - 127, -112), 127); }
// 2^e for e in [-127, 127] (2^-127 as zero).
__device__ __forceinline__ float pow2(int e) { return __builtin_bit_cast(float, (uint32_t)(e + 127) << 23); }

// x * sf (sf a power of two) as hi + lo.
__device__ __forceinline__ void split1(float x, float sf, _Float16 &hi, _Float16 &lo) {
    hi = (_Float16)__builtin_fmaf(x, sf, 0.f);
    lo = (_Float16)__builtin_fmaf(x, sf, -(float)hi);
}
__device__ __forceinline__ void split8(const float *x, float sf, v8h &hi, v8h &lo) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        hi[e] = (_Float16)__builtin_fmaf(x[e], sf, 0.f);
        lo[e] = (_Float16)__builtin_fmaf(x[e], sf, -(float)hi[e]);
    }
}

// max(|x|, |y|, m). Written out because fmaxf costs a canonicalising instruction more per value. NaNs are passed over.
__device__ __forceinline__ float max_abs2(float x, float y, float m) {
    float r;
    asm("v_max3_f32 %0, |%1|, |%2|, %3" : "=v"(r) : "v"(x), "v"(y), "v"(m));
    return r;
}
template <int N>
__device__ __forceinline__ float max_abs(const float *x) {
    static_assert(N % 2 == 0, "pairs");
    float m = 0.f;
#pragma unroll
    for (int e = 0; e < N; e += 2) m = max_abs2(x[e], x[e + 1], m);
    return m;
}
// The largest of the 16 lanes of a row of lanes, in each of them (the steps of wave_max, m >= 0). Written out: the
// compiler makes a move, a canonicalising maximum and the maximum of each step. (A permute reads its operand two wait
// states after the write.)
__device__ __forceinline__ float max16(float m) {
    asm("s_nop 1\n\tv_max_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_max_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf\n\ts_nop 0"
        : "+v"(m));
    return m;
}
// The bits of the largest of 64 non-negative values, wave-uniform (such floats order as their bits do).
__device__ __forceinline__ int wave_max_bits(float m) {
    const int v = __builtin_bit_cast(int, max16(m));
    return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}
// The wave's maxima of sixteen non-negative values: top[x] holds that of m[x + 4 y] in the lanes of row y (16 lanes). The halves
// of two registers trade places, then the rows, so that a step's maximum halves the number of registers: 12 swaps and 4 row
// maxima where one value after the other takes 16 of them.
__device__ __forceinline__ void wave_max_rows(const float *m, float *top) {
    uint32_t r[16];
#pragma unroll
    for (int x = 0; x < 16; ++x) r[x] = __builtin_bit_cast(uint32_t, m[x]);
#pragma unroll
    for (int x = 0; x < 8; ++x) {  // lanes 0 - 31: value x, 32 - 63: x + 8
        const auto v = __builtin_amdgcn_permlane32_swap(r[x], r[x + 8], false, false);
        r[x] = max(v[0], v[1]);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        const auto v = __builtin_amdgcn_permlane16_swap(r[x], r[x + 4], false, false);
        top[x] = max16(__builtin_bit_cast(float, max(v[0], v[1])));
    }
}
constexpr int kInfBits = 0x7f800000;

__device__ __forceinline__ v4f mfma_f16(v8h a, v8h b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
// c += a b of two split operands (the small products first).
__device__ __forceinline__ v4f mfma_split(v8h ah, v8h al, v8h bh, v8h bl, v4f c) {
    c = mfma_f16(al, bh, c);
    c = mfma_f16(ah, bl, c);
    return mfma_f16(ah, bh, c);
}

}  // namespace kea
