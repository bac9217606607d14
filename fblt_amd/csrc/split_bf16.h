/*
 * fp32 contractions on the bf16 matrix instructions: the operands as sums of lower-precision terms, the
 * products of the leading terms added in fp32 (the splitting of Dekker 1971, as used for matrix units by
 * Markidis et al. 2018 and Henry, Tang and Heinecke 2019, "Leveraging the bfloat16 artificial intelligence
 * datatype for higher-precision computations").
 *
 * An fp32 value is the exact sum of three bf16 values (each rounded to nearest from what the ones before leave; 8
 * significant bits each, 24 in all), as long as its last bit, a multiple of 2^-149 for any fp32 value, is at least
 * the smallest bf16 subnormal, 2^-133 (the matrix instructions take bf16 subnormals as they are).  Below 2^-110 the sum
 * is within 2^-134 only: products of operands of 1e-36 had a relative error of 2.7e-5.  So operands whose relative error
 * counts are taken times a power of two, and the results come out that much larger:
 *   - both operands of a plain product times SPLIT_UP, which makes the sum exact for every fp32 value;
 *   - in an attention the queries and the values times SPLIT_FAR, keys and weights as they are.  A key's error of
 *     2^-134 meets queries of at most 2^96 (larger ones overflow, see below): at most 2^-31 in a score, where the score's
 *     absolute error is what counts.  A weight's error of 2^-134 is below the 2^-126 at which the exponential unit cuts
 *     weights off.
 * SPLIT_DOWN takes either back.  A product of two such sums is taken as the six
 * partial products that are at least 2^-18 of it,
 *     x y = h h' + (h m' + m h') + (h l' + l h' + m m')  (+ m l' + l m' + l l', below 2^-25)
 * accumulated in fp32 by v_mfma_f32_32x32x16_bf16.  Against float64 the result is a little closer than
 * that of v_mfma_f32_32x32x2_f32, which rounds the accumulator eight times as often (2-norm of the
 * error over that of the result, K = 512, mixed signs: 3.3e-7 against 4.0e-7; with three products: 4e-6).
 * Six bf16 instructions take 192 cycles of the matrix unit where the fp32 ones take 512, and they leave
 * the vector ALU free, which the fp32 ones do not.
 *
 * A value that is not finite, or rounds to infinity in bf16 (above 3.39e38 with its factor), leaves NaN in the lower
 * parts and so in every result it takes part in; a result above 7.9e28 overflows before it is scaled back.  The
 * caller looks for results that are not finite and computes those on the fp32 instructions.
 */
#ifndef FBLT_AMD_SPLIT_BF16_H
#define FBLT_AMD_SPLIT_BF16_H

#include <hip/hip_runtime.h>

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr float SPLIT_UP = 0x1p16f, SPLIT_FAR = 0x1p32f, SPLIT_DOWN = 0x1p-32f;

/* N values -> their three parts.  (v_dot2_f32_bf16 would take a part off in one instruction instead of a shift or mask and
 * a subtraction, but it runs in the matrix unit's place: twelve matrix instructions, 179 ns alone, with eight of each in
 * between take 252 ns with conversions, 220 with shifts, 393 with it.) */
template <int N, typename Vec>
__device__ __forceinline__ void split_bf16(const float (&x)[N], Vec &high, Vec &mid, Vec &low) {
    uint32_t *const out[3] = {reinterpret_cast<uint32_t *>(&high), reinterpret_cast<uint32_t *>(&mid), reinterpret_cast<uint32_t *>(&low)};
#pragma unroll
    for (int i = 0; i < N; i += 2) {
        float a = x[i], b = x[i + 1];
#pragma unroll
        for (int part = 0; part < 3; part++) {
            uint32_t pair = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)a, (__bf16)b});
            asm("" : "+v"(pair)); /* one conversion of the pair: seen through, each half is converted once more on its own */
            out[part][i / 2] = pair;
            a -= __uint_as_float(pair << 16), b -= __uint_as_float(pair & 0xFFFF0000u);
        }
    }
}

/* ... of N consecutive ones of a register array, times `factor` */
template <int N, int M>
__device__ __forceinline__ void split_bf16_at(const float (&x)[M], int first, bf16x8 (&parts)[3], float factor = 1.0f) {
    float y[N];
#pragma unroll
    for (int i = 0; i < N; i++) y[i] = x[first + i] * factor;
    split_bf16<N>(y, parts[0], parts[1], parts[2]);
}

/* acc += A B over 16 of K, smallest partial products first */
template <typename Acc>
__device__ __forceinline__ Acc mfma_split(const bf16x8 (&a)[3], const bf16x8 (&b)[3], Acc acc) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[1], acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], acc, 0, 0, 0);
}

#endif /* FBLT_AMD_SPLIT_BF16_H */
