// Floats as sums of bf16 parts (conv_split.hip, matmul in gemm.hip).
#pragma once

#include "common.hpp"

namespace spk::kern {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Both operands are split after a scaling by 2^24 (exact): the lowest bit of
// the smallest float, 2^-149, is then above the smallest normal bf16, 2^-126,
// so that no part of any float is lost or denormal, and no product of parts
// that a float32 sum would show underflows.  Sums are scaled back once
// (2^-48); those that leave the float range scaled, from operands of 2^104 or
// sums of 2^80 on, are summed again without parts (parts_unfit).  Unscaled,
// operands below 2^-110 lost their last parts: weights of 1e-37 gave errors of
// 2e-4 and 2e-38 of 1e-3.  The scaling is one operation more an element than
// the split's 5.5: 14x14 3x3 layer at batch 64 105.3 -> 106.2 us, attention over
// 20x20 maps at batch 8 67.1 -> 68.0.
constexpr float kPartsScale = 0x1p24f;
constexpr float kPartsUnscale = 0x1p-48f;

// 2^24 x = hi + mid + lo: each the nearest bf16 of what the ones before leave,
// so the sum is exact (three 8-bit significands hold the 24 of a float) for
// |x| < 2^104.  Two elements at a time, packed low half first.
__device__ __forceinline__ void split_pair(float x0, float x1, unsigned &h, unsigned &m, unsigned &l) {
    x0 *= kPartsScale;
    x1 *= kPartsScale;
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
// rounding: an infinite operand (scaled, too) or product has parts of both
// signs, and gives a sum that is infinite or NaN.
__device__ __forceinline__ bool parts_unfit(float sum) { return !(__builtin_fabsf(sum) < __builtin_inff()); }

// A wave's 32x32 block of sums over k0 .. k1 - 1 in float32 multiply-adds, on
// the fp32 matrix cores, 32 k a round: the block again where parts_unfit() says
// so of one of its outputs.  load_a / load_b(k, v) give the lane's row / column
// (lane & 31) at k + 8 * (lane >> 5) + 0..7, zeros past the end, and are called
// up to 32 k past k1.  A 14x14 3x3 layer of 256 channels over 64 images, 109 us,
// takes 182 us with one NaN pixel and 270 with one image of them, where 10.7
// and 19 ms were spent when each lane summed its own outputs alone; a 512^3
// product 25 us, 47 with a NaN.
template <typename LoadA, typename LoadB>
__device__ __forceinline__ floatx16 block_sum_f32(int k0, int k1, const LoadA &load_a, const LoadB &load_b) {
    floatx16 s;
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = 0.0f;
    float a0[8], b0[8], a1[8], b1[8];
    load_a(k0, a0);
    load_b(k0, b0);
    for (int k = k0; k < k1; k += 32) {
        load_a(k + 16, a1);
        load_b(k + 16, b1);
#pragma unroll
        for (int j = 0; j < 8; j++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[j], b0[j], s, 0, 0, 0);
        load_a(k + 32, a0);
        load_b(k + 32, b0);
#pragma unroll
        for (int j = 0; j < 8; j++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[j], b1[j], s, 0, 0, 0);
    }
    return s;
}

}  // namespace spk::kern
