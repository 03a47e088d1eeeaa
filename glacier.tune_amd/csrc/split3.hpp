// split3.hpp -- fp32 operands on bf16 matrix cores without losing bits.
//
// x = h + m + l, each term the bf16 nearest to what is left: |m| <= 2^-8 |x|,
// |l| <= 2^-16 |x|, and the sum is x exactly (24 significant bits, for |x| >=
// 2^-110; below that the last terms reach bf16's subnormals).  A product a b
// is then the sum of nine bf16 products, each exact in fp32; the three
// smallest (a.m b.l, a.l b.m, a.l b.l: below 2^-23 |a b| together, of either
// sign) are left out, so a product is off by less than an fp32 rounding.  A
// bf16 MFMA does 16 times the products of an fp32 MFMA per cycle: six of them
// take 6/16 of its time.  Measured against 64-bit products over the projections'
// ranges (K 896-4096), fp32 results: 3.3e-7 to 7.5e-7 relative, where fp32
// MFMAs left 5.3e-7 to 1.1e-6 (fewer roundings: 16 products to a sum step).
// A non-finite x (or one that rounds to infinity) has no such split: set()
// reports it, and the caller takes fp32 products for those operands.
#pragma once

#include "attn_common.hpp"

namespace glacier {

#if defined(__HIP_DEVICE_COMPILE__)
// One MFMA operand of 8 floats as its three bf16 terms.
struct Split3 {
  bf16x8 h, m, l;
  // true if any of the 8 has no split (the terms are then meaningless)
  __device__ inline bool set(const float (&x)[8]) {
    float bad = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      h[e] = (bf16)x[e];
      const float r1 = x[e] - (float)h[e];
      m[e] = (bf16)r1;
      const float r2 = r1 - (float)m[e];
      l[e] = (bf16)r2;
      bad += r2;  // NaN once x - h is not finite
    }
    return bad != bad;
  }
};
#endif

}  // namespace glacier
