// float32 operands as three bfloat16 terms: x = h + m + l exactly (8 + 8 + 8
// significant bits, each term the nearest-even rounding of what is left), so
// that the bf16 matrix cores, 16 times the float32 ones' rate on gfx950,
// multiply float32 values: of the nine products of two such triples the six
// of at least 2^-16 of the largest are kept (hh, hm, mh, hl, mm, lh), which
// drops at most 2^-24 of |x y| per product, one float32 rounding. Operands
// past bf16's largest finite value, infinities and NaNs give NaN.
#ifndef VOXCPM_AMD_BF16X3_HPP_
#define VOXCPM_AMD_BF16X3_HPP_

#include <hip/hip_runtime.h>

#include <cstdint>

#include "q8.hpp"
#include "q8_tile.hpp"

namespace vx::bf16x3 {

typedef float F32x16 __attribute__((ext_vector_type(16)));

/// C (32 x 32, float32) += A (32 x 16, bf16) B (16 x 32, bf16): lane L holds
/// A row L % 32 and B column L % 32, each at reduction indices
/// 8 (L / 32) .. + 7; C element v of lane L is row 8 (v / 4) + 4 (L / 32) +
/// v % 4, column L % 32.
__device__ inline F32x16 Mfma32(const q8::Bf16x8& a, const q8::Bf16x8& b, const F32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

/// The terms of two values, each packed low / high.
struct Pair {
  std::uint32_t h, m, l;
};

__device__ inline Pair Split(float lo, float hi) {
  Pair out;
  out.h = q8::PackBf16x2(lo, hi);
  lo -= q8::Bf16Lo(out.h);
  hi -= q8::Bf16Hi(out.h);
  out.m = q8::PackBf16x2(lo, hi);
  lo -= q8::Bf16Lo(out.m);
  hi -= q8::Bf16Hi(out.m);
  out.l = q8::PackBf16x2(lo, hi);
  return out;
}

/// The terms of eight values as three MFMA operands.
struct Octet {
  uint4 h, m, l;
};

__device__ inline Octet Split(const float4& a, const float4& b) {
  const Pair p0 = Split(a.x, a.y);
  const Pair p1 = Split(a.z, a.w);
  const Pair p2 = Split(b.x, b.y);
  const Pair p3 = Split(b.z, b.w);
  return Octet{uint4{p0.h, p1.h, p2.h, p3.h}, uint4{p0.m, p1.m, p2.m, p3.m},
               uint4{p0.l, p1.l, p2.l, p3.l}};
}

}  // namespace vx::bf16x3

#endif  // VOXCPM_AMD_BF16X3_HPP_
