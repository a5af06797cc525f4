// float32 products on gfx950's f16 matrix cores: x = h + l / 2048 with h and
// l the nearest-even float16 of x and of 2048 (x - h), 22 significant bits
// and more (the residual's sign is one). Of the four products of two such
// pairs the three of at least 2^-11 of the largest are kept, hh and the
// cross terms hl + lh, which sum apart and join the first scaled by 2^-11.
// Against the float32 matrix instructions, a sixteenth of the f16 rate, the
// operands lose at most two bits, and the sums round once per 16 terms
// instead of once per 4, which more than makes up for it over long
// reductions. Below 2^-14 h turns subnormal and l takes over what it drops,
// in steps of 2^-35: an absolute error of at most 2^-36 per operand, whatever
// its size, so that operands which are small throughout would lose float32's
// precision. From 65520 on h is infinite and l is too, of the other sign: a sum
// with such an operand is NaN, whatever it is multiplied by. Callers start
// over in a format of float32's range (three bfloat16 terms, bf16x3.hpp, or
// float32 itself) where a group of operands is neither zeros nor large enough
// (Least), and where an operand is too large (TooLarge, or by the NaN).
#ifndef VOXCPM_AMD_F16X2_HPP_
#define VOXCPM_AMD_F16X2_HPP_

#include <hip/hip_runtime.h>

#include <cstdint>

#include "bf16x3.hpp"

namespace vx::f16x2 {

using bf16x3::F32x16;
typedef _Float16 F16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 F16x2 __attribute__((ext_vector_type(2)));
typedef float F32x2 __attribute__((ext_vector_type(2)));

constexpr float kLargest = 65504.0F;
constexpr float kResidual = 2048.0F;       // the residual's scale
constexpr float kCross = 1.0F / kResidual;  // the cross terms'

__device__ inline F16x8 AsF16x8(const uint4& bits) { return __builtin_bit_cast(F16x8, bits); }

/// C (32 x 32, float32) += A (32 x 16, f16) B (16 x 32, f16), the lanes'
/// layout that of bf16x3::Mfma32.
__device__ inline F32x16 Mfma32(const uint4& a, const uint4& b, const F32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(AsF16x8(a), AsF16x8(b), c, 0, 0, 0);
}

/// The terms of two values, each packed low / high.
struct Pair {
  std::uint32_t h, l;
};

__device__ inline Pair Split(float lo, float hi) {
  const F16x2 h = __builtin_convertvector((F32x2{lo, hi}), F16x2);
  // One rounding each: 2048 lo and 2048 h are exact, as is their difference.
  const F16x2 l = {
      static_cast<_Float16>(__builtin_fmaf(static_cast<float>(h.x), -kResidual, lo * kResidual)),
      static_cast<_Float16>(__builtin_fmaf(static_cast<float>(h.y), -kResidual, hi * kResidual))};
  return Pair{__builtin_bit_cast(std::uint32_t, h), __builtin_bit_cast(std::uint32_t, l)};
}

/// The terms of eight values as two MFMA operands.
struct Octet {
  uint4 h, l;
};

__device__ inline Octet Split(const float4& a, const float4& b) {
  const Pair p0 = Split(a.x, a.y);
  const Pair p1 = Split(a.z, a.w);
  const Pair p2 = Split(b.x, b.y);
  const Pair p3 = Split(b.z, b.w);
  return Octet{uint4{p0.h, p1.h, p2.h, p3.h}, uint4{p0.l, p1.l, p2.l, p3.l}};
}

/// max(most, |v|) over the components (NaNs pass by: their terms are NaNs).
__device__ inline float Largest(float most, const float4& v) {
  most = fmaxf(fmaxf(most, fabsf(v.x)), fabsf(v.y));
  return fmaxf(fmaxf(most, fabsf(v.z)), fabsf(v.w));
}
__device__ inline bool TooLarge(float most) { return most > kLargest; }

/// The smallest nonzero one of the groups' largest magnitudes: the error of
/// a small operand, at most 2^-36, is at most 2^-36 / least of its group's
/// largest.
struct Least {
  std::uint32_t bits = ~0U;  // the magnitude's bits less one: zero comes last
  __device__ void Add(float group) {
    const std::uint32_t own = __builtin_bit_cast(std::uint32_t, group) - 1U;
    bits = own < bits ? own : bits;
  }
  __device__ bool Below(float limit) const {
    return bits < __builtin_bit_cast(std::uint32_t, limit) - 1U;
  }
};

/// The groups' Least and the largest magnitude of all.
struct Range {
  float most = 0.0F;
  Least least;
  __device__ void Add(float group) {
    most = fmaxf(most, group);
    least.Add(group);
  }
  __device__ bool Holds(float at_least) const {
    return !TooLarge(most) && !least.Below(at_least);
  }
};

}  // namespace vx::f16x2

#endif  // VOXCPM_AMD_F16X2_HPP_
