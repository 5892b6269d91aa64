// fp32 operands on the 16-bit matrix cores: x = h + m + l, three bf16 parts, each the rounded remainder of those before it
// (8 + 8 + 8 significant bits: nothing is left of a 24-bit significand), and
//   a b = ah bh + (ah bm + am bh + am bm + ah bl + al bh),
// six exact products per pair; what is left out (am bl, al bm, al bl) is below 2^-24.1 of the product, 2^-27.5 in the mean (a sum of one
// product is off by up to 0.97 units in the last place, rounded once by 0.5; sums gain, see below).  The first sum and that of
// the five small terms have an accumulator each: the small ones' roundings then fall 2^-8 below those of the first, which has one
// rounding per 16 contraction indexes where v_mfma_f32_32x32x2_f32 has one per 2.  Measured against 64 bits, relative 2-norm, normal
// operands (the fp32 instruction on the same operands): contraction of 16 3.5e-8 (8.0e-8), 256 9.1e-8 (3.0e-7), 5248 4.6e-7
// (1.3e-6), 24000 1.0e-6 (2.8e-6); with one accumulator for all six 3.3e-8, 2.4e-7, 1.1e-6, 2.5e-6.
// The matrix pipe takes six such products in 3/8 of the fp32 instruction's time (16 times its rate).
//
// Infinities, NaN and magnitudes that round to infinity in bf16 leave NaN in a part, and so in every result that they
// reach.  Magnitudes below 2^-110 lose their last bits to the parts' underflow: 2^-134 absolute (subnormal parts are kept),
// times the other operand, which only a small result can feel.  So the kernels compute what a wave holds a second time, on the fp32
// instruction, where a result is not finite, or not zero and below 2^-90.  What is left of the underflow is below 2^-24 of a result as
// long as the other operand's magnitudes add up to no more than 2^20 over the contraction, and operands below 2^-134 count as zero where all
// results that they reach are zero with them (zeros alone are not looked at again: masks and padding are full of them).  (Measured before the second condition: operands
// of 2^-115 1.1e-6, of 2^-126 2.2e-3 in the 2-norm, the fp32 instruction 4e-7.)  It takes 3 to 5 times as long as the first where one
// infinity reaches every tile, up to 9 times where all results are small: 3 x 3, 256 -> 256 channels over 14 x 14, 64 images 95 us -> 388,
// 611 in all, 21 taps, 250 -> 250 channels, 16 x 1500 frames 289 -> 1623, 2840.
#pragma once
#include "conv2d_mfma.h"

namespace flhip {

// the parts of two neighbouring values, packed as bf16 pairs
struct Split2 {
  uint32_t h, m, l;
};
__device__ __forceinline__ Split2 split2(float x, float y) {
  Split2 s;
  s.h = pack_bf16(x, y);
  x -= __uint_as_float(s.h << 16);
  y -= __uint_as_float(s.h & 0xffff0000u);
  s.m = pack_bf16(x, y);
  x -= __uint_as_float(s.m << 16);
  y -= __uint_as_float(s.m & 0xffff0000u);
  s.l = pack_bf16(x, y);
  return s;
}

// big += ah bh, small += the other five; parts 0, 1, 2 = h, m, l
template <typename V>
__device__ __forceinline__ void split_mma(floatx16& big, floatx16& small, const V (&a)[3], const V (&b)[3]) {
  small = Lo16<bf16_t>::mma32(a[2], b[0], small);
  small = Lo16<bf16_t>::mma32(a[0], b[2], small);
  small = Lo16<bf16_t>::mma32(a[1], b[1], small);
  small = Lo16<bf16_t>::mma32(a[1], b[0], small);
  small = Lo16<bf16_t>::mma32(a[0], b[1], small);
  big = Lo16<bf16_t>::mma32(a[0], b[0], big);
}

// whether a result has to be computed a second time
__device__ __forceinline__ bool split_redo(float v) {
  const uint32_t u = __float_as_uint(v) & 0x7fffffffu;
  return u >= 0x7f800000u || u - 1u < 0x12800000u - 1u;      // (0x12800000 = 2^-90)
}

}  // namespace flhip
