// split3.hpp -- fp32 operands on bf16 matrix cores without losing bits.
//
// x = h + m + l, each term the bf16 nearest to what is left: |m| <= 2^-8 |x|,
// |l| <= 2^-17 |x|, and the sum is x exactly (24 significant bits) while the
// last term's bits lie above 2^-133, bf16's smallest subnormal: always for |x|
// >= 2^-110, below that for values with fewer bits (bf16 values among them).
// A product a b is then the sum of nine bf16 products, each exact in fp32 (MFMAs
// keep subnormals); the three smallest (a.m b.l, a.l b.m, a.l b.l) are left
// out: at most (2^-24 + 2^-34) |a b| together, an fp32 rounding.  A
// bf16 MFMA does 16 times the products of an fp32 MFMA per cycle: six of them
// take 6/16 of its time.  The five small products have a sum of their own, so
// that the large one's rounds once for 16 products.  Against 64-bit products over
// the projections' ranges (K 896-4096, T 60-540), fp32 results are 1.5e-7 to
// 3.9e-7 off in the 2-norm, where fp32 MFMAs left 3.3e-7 to 9.5e-7 (and all six in
// one sum 3.6e-7 to 9.7e-7).
// An x that is not that sum (not finite, rounding to infinity, or with bits
// below 2^-133) has no split: SplitMarks tell, and the caller takes fp32
// products for those operands.
#pragma once

#include "attn_common.hpp"

namespace glacier {

#if defined(__HIP_DEVICE_COMPILE__)
// Whether every float split since its start has a split: what is left for l is
// NaN once x - h is not finite, and otherwise a bf16 value unless its lower 16
// bits say otherwise.
struct SplitMarks {
  float sum = 0.0f;
  unsigned bits = 0;
  __device__ inline bool bad() const { return sum != sum || (bits & 0xffffu) != 0; }
};
// One MFMA operand of 8 floats as its three bf16 terms (meaningless for those
// without a split).
struct Split3 {
  bf16x8 h, m, l;
  __device__ inline void set(const float (&x)[8], SplitMarks& mark) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      h[e] = (bf16)x[e];
      const float r1 = x[e] - (float)h[e];
      m[e] = (bf16)r1;
      const float r2 = r1 - (float)m[e];
      l[e] = (bf16)r2;
      mark.sum += r2;
      mark.bits |= __float_as_uint(r2);
    }
  }
};
#endif

}  // namespace glacier
