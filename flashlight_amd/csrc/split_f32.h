// fp32 operands on the 16-bit matrix cores: x = h + m + l, three bf16 parts, each the rounded remainder of those before it
// (8 + 8 + 8 significant bits: nothing is left of a 24-bit significand), and
//   a b = ah bh + (ah bm + am bh + am bm + ah bl + al bh),
// six exact products per pair; what is left out (am bl, al bm, al bl) is below 2^-26 of the product.  The first sum and that of
// the five small terms have an accumulator each: the small ones' roundings then fall 2^-8 below those of the first, which has one
// rounding per 16 contraction indexes where v_mfma_f32_32x32x2_f32 has one per 2.  Measured against 64 bits, relative 2-norm, normal
// operands (the fp32 instruction on the same operands): contraction of 16 3.5e-8 (8.0e-8), 256 9.1e-8 (3.0e-7), 5248 4.6e-7
// (1.3e-6), 24000 1.0e-6 (2.8e-6); with one accumulator for all six 3.3e-8, 2.4e-7, 1.1e-6, 2.5e-6.
// The matrix pipe takes six such products in 3/8 of the fp32 instruction's time (16 times its rate).
//
// Infinities, NaN and magnitudes that round to infinity in bf16 leave NaN in a part, and so in every result that they
// reach: the kernels compute tiles with a result that is not finite a second time, on the fp32 instruction.  Magnitudes below
// 2^-110 lose their last bits to the parts' underflow (2^-134 absolute).
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

__device__ __forceinline__ bool not_finite(float v) { return (__float_as_uint(v) & 0x7f800000u) == 0x7f800000u; }

}  // namespace flhip
