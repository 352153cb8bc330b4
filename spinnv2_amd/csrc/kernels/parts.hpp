// Floats as sums of bf16 parts (conv_split.hip, matmul in gemm.hip).
#pragma once

#include "common.hpp"

namespace spk::kern {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// x = hi + mid + lo: each the nearest bf16 of what the ones before leave, so
// the sum is x exactly (three 8-bit significands hold the 24 of a float).
// Two elements at a time, packed low half first.
__device__ __forceinline__ void split_pair(float x0, float x1, unsigned &h, unsigned &m, unsigned &l) {
    h = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{x0, x1}, bf16x2));
    const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
    m = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{r0, r1}, bf16x2));
    const float s0 = r0 - __uint_as_float(m << 16), s1 = r1 - __uint_as_float(m & 0xffff0000u);
    l = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{s0, s1}, bf16x2));
}

// Fewest products a sum on parts takes the place of float32 multiply-adds for:
// the three part products left out and the part sums' own roundings stay within
// what multiply-adds round from three on (largest error relative to sum |ab|,
// in 2^-24, multiply-adds against parts: K = 1 1.00 and 1.59, 2 1.94 and 2.65,
// 3 2.45 and 2.12, 16 4.4 and 1.9).
constexpr int kPartsMinK = 3;

// Whether a sum of part products may differ from the float32 sum by more than
// rounding: an infinite input or product has parts of both signs, and the
// parts of values near the smallest float round to zero.
__device__ __forceinline__ bool parts_unfit(float sum) {
    const float v = __builtin_fabsf(sum);
    return !(v < __builtin_inff()) || (v < 0x1p-90f && v != 0.0f);
}

}  // namespace spk::kern
