/*
 * fp32 contractions on the f16 matrix instructions: each operand as a sum of two f16 values, for operands whose range the
 * caller has looked at.  Half the matrix instructions of the three bf16 parts of split_bf16.h, half the conversions, and
 * less power, which is what the clock follows where the matrix unit works without a pause.
 *
 * x = high + low, each rounded to nearest: what high leaves is at most 2^12 units in the last place of x, and low holds 11
 * bits of it, so the sum is x itself or, where the rest is odd and above 2^11, one unit in the last place off (a quarter of
 * all values).  f16 ends at 2^16 and at 2^-24, so `low` is kept times HALF_UP: then a value of at least 2^-14 is as close as
 * that, and a smaller one within 2^-36.  half_range() says whether a run of values may be taken so: all zero, or the largest
 * between 2^-13 and 2^16.  A product is
 *     x y = h h' + (h l' 2^11 + l 2^11 h') 2^-11      (+ l l', below 2^-22 and of either sign)
 * with the small products in an accumulator of their own, or, where one operand stays and can be scaled by its owner so that
 * its largest value is near 2^15, h h' + h l' + (l 2^11) (h' 2^-11) in one: what that loses of the owner's small values
 * is below 2^-40 of the largest.  Small products first, or apart, the sum of the large ones is rounded once for 16 terms, not
 * six times as with bf16 parts: attention over 32 problems of 4096 rows has 0.55 of its error against float64, over 300
 * rows 0.87, never more (2-norm; 40 shapes and scales).
 */
#ifndef FBLT_AMD_SPLIT_F16_H
#define FBLT_AMD_SPLIT_F16_H

#include <hip/hip_runtime.h>

typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

constexpr float HALF_UP = 0x1p11f, HALF_DOWN = 0x1p-11f;

/* two values as f16 */
__device__ __forceinline__ halfx2 half_pair(float a, float b) {
    halfx2 p = {(_Float16)a, (_Float16)b};
    asm("" : "+v"(p)); /* one conversion of the pair */
    return p;
}

/* what the halves of p leave of a and b: exact; one mixed multiply-add each (seen through, -1 makes it a conversion and a
 * subtraction) */
__device__ __forceinline__ void half_rest(halfx2 p, float &a, float &b) {
    float minus = -1.0f;
    asm("" : "+v"(minus));
    a = __builtin_fmaf((float)p.x, minus, a);
    b = __builtin_fmaf((float)p.y, minus, b);
}

/* N values -> high, and what it leaves times HALF_UP */
template <int N, typename Vec>
__device__ __forceinline__ void split_f16(const float (&x)[N], Vec &high, Vec &low) {
    halfx2 *const to[2] = {reinterpret_cast<halfx2 *>(&high), reinterpret_cast<halfx2 *>(&low)};
#pragma unroll
    for (int i = 0; i < N; i += 2) {
        float a = x[i], b = x[i + 1];
        const halfx2 p = half_pair(a, b);
        half_rest(p, a, b);
        to[0][i / 2] = p;
        to[1][i / 2] = half_pair(a * HALF_UP, b * HALF_UP);
    }
}

/* N values -> high, what it leaves, and high times HALF_DOWN */
template <int N, typename Vec>
__device__ __forceinline__ void split_f16_down(const float (&x)[N], Vec &high, Vec &low, Vec &down) {
    halfx2 *const to[3] = {reinterpret_cast<halfx2 *>(&high), reinterpret_cast<halfx2 *>(&low), reinterpret_cast<halfx2 *>(&down)};
#pragma unroll
    for (int i = 0; i < N; i += 2) {
        float a = x[i], b = x[i + 1];
        const halfx2 p = half_pair(a, b);
        half_rest(p, a, b);
        to[0][i / 2] = p;
        to[1][i / 2] = half_pair(a, b);
        to[2][i / 2] = p * halfx2{(_Float16)HALF_DOWN, (_Float16)HALF_DOWN};
    }
}

/* may these values be the stored side?  (A NaN passes, and shows in the result.) */
template <int N>
__device__ __forceinline__ bool half_range(const float (&x)[N]) {
    float top = 0.f;
#pragma unroll
    for (int i = 0; i < N; i++) top = fmaxf(top, fabsf(x[i]));
    return (top == 0.f) | ((top >= 0x1p-13f) & (top < 65504.f));
}

/* acc += A B over 16 of K */
template <typename Acc, typename VecA, typename VecB>
__device__ __forceinline__ Acc mfma_f16(const VecA &a, const VecB &b, Acc acc) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, b), acc, 0, 0, 0);
}

#endif /* FBLT_AMD_SPLIT_F16_H */
