// Snake, the AudioVAE decoder's activation.
#ifndef VOXCPM_AMD_SNAKE_HPP_
#define VOXCPM_AMD_SNAKE_HPP_

#include <hip/hip_runtime.h>

namespace vx {

/// A channel's 1 / (a + 1e-9) in Snake.
__device__ inline float SnakeScale(float a) { return 1.0F / (a + 1e-9F); }
/// Snake(y) = y + sin^2(a y) / (a + 1e-9), `inverse` the channel's
/// SnakeScale(a). The sine is the hardware's (v_sin_f32 takes turns:
/// sin(2 pi r)) of a y in turns reduced to [-1/2, 1/2]: the decoder
/// evaluates Snake on every element of every unit and block input, and the
/// library sine's range reduction and polynomial made the units' products
/// bound by their vector instructions.
__device__ inline float Snake(float y, float a, float inverse) {
  const float turns = a * y * 0.159154943091895336F;  // 1 / (2 pi)
  const float s = __builtin_amdgcn_sinf(turns - rintf(turns));
  return y + inverse * (s * s);
}
__device__ inline float Snake(float y, float a) { return Snake(y, a, SnakeScale(a)); }

/// A channel's constants where many elements share them: a / (2 pi), and
/// 1 / (a + 1e-9) by the hardware's reciprocal and one Newton step (a
/// twelfth of a residual unit's vector instructions were its divisions).
struct SnakeChannel {
  float turns = 0.0F;
  float inverse = 0.0F;
  SnakeChannel() = default;
  __device__ explicit SnakeChannel(float a) : turns(a * 0.159154943091895336F) {
    const float x = a + 1e-9F;
    const float r = __builtin_amdgcn_rcpf(x);
    inverse = __builtin_fmaf(__builtin_fmaf(-x, r, 1.0F), r, r);
  }
  __device__ float operator()(float y) const {
    const float t = turns * y;
    const float s = __builtin_amdgcn_sinf(t - rintf(t));
    return y + inverse * (s * s);
  }
};

}  // namespace vx

#endif  // VOXCPM_AMD_SNAKE_HPP_
