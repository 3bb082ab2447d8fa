// fp32 products on the fp16 matrix cores.
//
// A number x is taken as hi + lo / 2048: hi is x rounded to half precision, lo the rest times 2048 rounded to half precision (the
// factor keeps it among half's normal numbers), together 22 bits and a sign (the split of Ootomo and Yokota, "Recovering single
// precision accuracy from Tensor Cores while surpassing the FP32 theoretical peak performance", 2022).  Of a product of two such numbers
//     hi hi  +  (hi lo + lo hi) / 2048
// is formed, each partial product exact in the matrix core; what is left out (lo lo) and what the rounding of lo takes are at most
// 2^-22 of the product, of either sign, and smaller still against a sum of many.  The two parts have an accumulator each: one
// instruction then adds 16 products to a running sum that is rounded once, where the fp32 instruction adds two, so that a sum over
// 768 is rounded 48 times instead of 384, and the whole comes out closer to 64 bits than on the fp32 matrix cores.  Three
// instructions of v_mfma_f32_32x32x16_f16 take 3/16 of the time of the fp32 ones (peaks of 2.5 against 0.157 PFLOP/s; a large
// half-precision product is held to 1.2 by the card's power).  Three bfloat16 terms have fp32's range but need six instructions.
//
// Half precision's range: hi is off by less than 2^-12 of x from 6e-5 to 65504 and both together by less than 2^-36 below.  So what
// goes in is scaled by powers of two (exact) to a size around 1, and what does not fit all the same comes out as an infinity or NaN:
// linear.hip and attention.hip look at their results and form the ones that are not finite again in plain fp32.  bh4_split.hip and
// fht_bwd.hip scale by a row's largest number, so that a finite row fits; one with an infinity or NaN comes out as NaN, by itself.
#pragma once

#include "lffn_common.h"

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr float SPLIT_LO = 2048.f;

// Two numbers times `scale` (a power of two) as a packed pair of hi and one of lo.
__device__ __forceinline__ uint32_t split_hi(float a, float b, float scale) {
    const f32x2_t v = {a * scale, b * scale};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
}
__device__ __forceinline__ uint32_t split_lo(float a, float b, float scale, uint32_t hi) {
    const f16x2_t h = __builtin_bit_cast(f16x2_t, hi);
    const float s = scale * SPLIT_LO;
    const f32x2_t v = {fmaf((float)h[0], -SPLIT_LO, a * s), fmaf((float)h[1], -SPLIT_LO, b * s)};      // exact
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
}

// lo without the factor, of two numbers that are large enough for it to be among half's normal numbers (their largest 2^6 and more)
__device__ __forceinline__ uint32_t split_rest(float a, float b, uint32_t hi) {
    f32x2_t v;
    // a - hi (exact), the half-precision operand widened inside the instruction: the compiler forms a conversion and a subtraction
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(v[0]) : "v"(hi), "v"(a));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(v[1]) : "v"(hi), "v"(b));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
}

__device__ __forceinline__ f32x16_t mfma_f16(uint4 a, uint4 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// Row (of the A operand) that element i of a lane's 32 x 32 result belongs to; the column (of the B operand) is lane % 32.  The
// operands: row or column lane % 32, k = 8 (lane / 32) ... + 7.
__host__ __device__ __forceinline__ constexpr int mfma_row(int i, int half) { return 8 * (i / 4) + 4 * half + i % 4; }

__device__ __forceinline__ bool is_finite(float v) { return (__float_as_uint(v) & 0x7F800000u) != 0x7F800000u; }

// The power of two that takes numbers of largest magnitude `most` to [1, 2), and its inverse; 1 where there is none.
struct PowerOfTwo {
    float scale, inverse;
};
__device__ __forceinline__ PowerOfTwo scale_to_one(float most) {
    uint32_t e = (__float_as_uint(most) >> 23) & 0xFFu;
    e = e == 0 || e == 255 ? 127 : min(max(e, 16u), 252u);          // (times or by 2^15 still a normal number)
    return {__uint_as_float((254 - e) << 23), __uint_as_float(e << 23)};
}

// The power of two that takes numbers of largest magnitude `most`, or a sample's, to [2^top, 2^(top + 1)); `exponent` is that of the way
// back.  A number is then held to 22 bits down to 2^-(14 + top) of that largest one and a smaller one to 2^-(36 + top) of it (lo without
// its factor: 2^-(3 + top) and 2^-(25 + top)).  Nothing but zeros, or numbers below 2^-103, is scaled as 2^-103 would be, so that a sample
// of zeros hides no small numbers behind it: they outgrow it.
__device__ __forceinline__ float scale_to(float most, int top, int &exponent) {
    const int bits = __float_as_uint(most) >> 23, e = bits == 255 ? 127 : max(bits, 24);     // (times 2048 still a number)
    exponent = e - 127 - top;
    return __uint_as_float((254 - e + top) << 23);
}

// Largest over the four rows of 16 lanes (row swaps on the vector ALU: an LDS permute would be waited for).
__device__ __forceinline__ float rows_most(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// A barrier behind the LDS accesses issued so far; global loads stay in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
