// The AudioVAE decoder's products over many rows (a whole utterance) on the
// f16 matrix cores with float32 operands as two float16 terms (f16x2.hpp;
// operands outside their range as three bfloat16 ones, bf16x3.hpp), and its
// residual units of 32 and 64 channels as one launch each (vae_wide.hip).
#ifndef VOXCPM_AMD_VAE_WIDE_HPP_
#define VOXCPM_AMD_VAE_WIDE_HPP_

#include <hip/hip_runtime.h>

#include <cstddef>

namespace vx::vae {

/// What becomes of v = product + bias (+ the stream's value): the stream's
/// new value (kStream); the next block's input Snake(v scale + shift, alpha)
/// (kBlockInput: rows [1 + t] with the last chunk's final row first); or the
/// output window Snake(v, alpha) (kOutput: rows [6 + t], the last chunk's
/// final six first).
enum class Target : int { kStream = 0, kBlockInput = 1, kOutput = 2 };

struct Epilogue {
  Target target = Target::kStream;
  const float* bias = nullptr;   // [channels], output column n at n % channels
  int channels = 1;
  const float* prior = nullptr;  // [t][n] added to the product, or null
  float* out = nullptr;          // [t][n], or the target's rows
  const float* scale = nullptr;  // [n]: kBlockInput
  const float* shift = nullptr;
  const float* alpha = nullptr;  // [n]: kBlockInput, kOutput
  // kBlockInput, kOutput: the history rows before the first output row, and
  // (kBlockInput) where the last output row is left for the next chunk.
  const float* history = nullptr;
  float* history_next = nullptr;
};

/// y = epilogue(A W^T): A's row f is x[f][0 .. k), or (taps) the
/// block input's pair [u(f) | u(f - 1)] of k / 2 channels each from rows
/// u(-1), u(0), .. at x. W [n][k]. k a multiple of 32 (taps: of 64).
struct Product {
  const float* x = nullptr;
  const float* w = nullptr;
  bool taps = false;
  float* tail = nullptr;  // when set, receives x's last row's first k / 2 values
  int t = 0;
  int k = 0;
  int n = 0;
  Epilogue epilogue;
};

void RunProduct(const Product& p, hipStream_t stream);

/// A residual unit's Snake and dilated depthwise convolution: the stream's
/// rows y [t][c], the last chunk's 6 d rows of Snake(y) in `state`, and
/// where this chunk's are left (t >= 6 d).
struct Unit {
  const float* y = nullptr;
  const float* alpha_in = nullptr;
  const float* taps = nullptr;  // [c][7]
  const float* bias = nullptr;
  const float* alpha_out = nullptr;
  const float* state = nullptr;
  float* state_next = nullptr;
  int t = 0;
  int c = 0;
  int d = 1;  // 1, 3 or 9
};

/// out [t][c] = Snake(depthwise(Snake(y))), a product's operand.
void RunDepthwise(const Unit& u, float* out, hipStream_t stream);

/// Whether RunUnit takes units of c channels.
bool UnitSupported(std::size_t c);
/// The whole unit: epilogue(Snake(depthwise(Snake(y))) W^T), W [c][c].
/// epilogue.out must not be y.
void RunUnit(const Unit& u, const float* w, const Epilogue& epilogue, hipStream_t stream);

}  // namespace vx::vae

#endif  // VOXCPM_AMD_VAE_WIDE_HPP_
