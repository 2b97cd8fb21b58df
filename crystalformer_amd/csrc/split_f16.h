// fp32 products on the f16 matrix instructions: both factors as two halves of 11 bits, x 2^k = hi + lo, and all four
// products summed in fp32.  Scaled so that the largest value lies in [2^14, 2^15) a value keeps 22 bits and a sign down to
// 2^-16 of it and is off by up to 2^-39 of it below (a half's last bit is 2^-24).  v_mfma_f32_16x16x32_f16 runs beside vector instructions (17 cycles; eight
// v_fma beside it 36, 22 without it) where v_mfma_f32_16x16x4_f32 holds them up (32 cycles; 57 with the same eight).
#pragma once
#include "cf_common.h"

namespace cf {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef int int4_t __attribute__((ext_vector_type(4)));
typedef int int2_t __attribute__((ext_vector_type(2)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// x0, x1 times `scale` as two halves each, packed in pairs.
struct Split2 {
    int hi, lo;
};
__device__ __forceinline__ Split2 split2(float x0, float x1, float scale, float zero)
{
    half2_t h = {(_Float16)__builtin_fmaf(x0, scale, zero), (_Float16)__builtin_fmaf(x1, scale, zero)};
    Split2 s;
    s.hi = __builtin_bit_cast(int, h);
    asm("" : "+v"(s.hi));                   // (one packed register: else the second half is worked out twice)
    h = __builtin_bit_cast(half2_t, s.hi);
    const half2_t l = {(_Float16)__builtin_fmaf(x0, scale, -(float)h[0]), (_Float16)__builtin_fmaf(x1, scale, -(float)h[1])};
    s.lo = __builtin_bit_cast(int, l);
    return s;
}

// The same with the second halves scaled by 2^11 beyond the first, for values that share a scale with others of any size: of
// values scaled by 2^26 (the largest in [2^25, 2^26)) one keeps 22 bits and a sign down to 2^-27 of the largest and is off by up
// to 2^-50 of it below.  The products of each kind of halves are summed apart (sum_of_kinds), which a long sum wants anyway:
// every addition to the large sum rounds it.
constexpr float LO_SCALE = 2048.0f;
__device__ __forceinline__ Split2 split2_far(float y0, float y1, float zero)
{
    half2_t h = {(_Float16)__builtin_fmaf(y0, 1.0f / LO_SCALE, zero), (_Float16)__builtin_fmaf(y1, 1.0f / LO_SCALE, zero)};
    Split2 s;
    s.hi = __builtin_bit_cast(int, h);
    asm("" : "+v"(s.hi));                   // (as above)
    h = __builtin_bit_cast(half2_t, s.hi);
    const half2_t l = {(_Float16)__builtin_fmaf((float)h[0], -LO_SCALE, y0), (_Float16)__builtin_fmaf((float)h[1], -LO_SCALE, y1)};
    s.lo = __builtin_bit_cast(int, l);
    return s;
}
// (An infinite value's second half is not a number, and an infinity times a second half has any sign: the first halves' product
// is fp32's answer then, the rest is kept finite.  Of finite values the rest is below 2^60.)
__device__ __forceinline__ float4_t sum_of_kinds(float4_t hh, float4_t hl, float4_t lh, float4_t ll)
{
    float4_t r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float rest = __builtin_fmaf(ll[i], 1.0f / LO_SCALE, hl[i] + lh[i]);
        r[i] = __builtin_fmaf(__builtin_amdgcn_fmed3f(rest, -0x1p100f, 0x1p100f), 1.0f / LO_SCALE, hh[i]);
    }
    return r;
}

// (The exponent of a group of values is that of its largest finite one: beside an infinity's own the others would leave a
// half's range.)
__device__ __forceinline__ float finite_magnitude(float x) { return fabsf(x) < __builtin_inff() ? fabsf(x) : 0.f; }

__device__ __forceinline__ float4_t mfma16(int2_t a, int2_t b, float4_t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(half4_t, a), __builtin_bit_cast(half4_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ float4_t mfma32(int4_t a, int4_t b, float4_t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
}

__device__ __forceinline__ float rows_max(float v)
{
    unsigned x = (unsigned)__float_as_int(v);
    uint2_cf r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    v = fmaxf(__int_as_float((int)r[0]), __int_as_float((int)r[1]));
    x = (unsigned)__float_as_int(v);
    r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return fmaxf(__int_as_float((int)r[0]), __int_as_float((int)r[1]));
}

}  // namespace cf
