// Products of more than 128 activation rows whose weights go from their
// panels straight into the matrix cores' operands (q8_prefill.hip): the
// stacks' prefill products with their consumers' work in the epilogue, and
// the larger standalone ones.
#ifndef VOXCPM_AMD_Q8_PREFILL_HPP_
#define VOXCPM_AMD_Q8_PREFILL_HPP_

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "common.hpp"

namespace vx::prefill {

enum class Out : int {
  kStore = 0,       // y = product
  kAccumulate = 1,  // y += product
  kBf16 = 2,        // out = bf16(product)
  kSwiGlu = 3,      // out [m][n / 2] = bf16(silu(gate) up), n / 2 columns each
  kQkvCache = 4     // rotary embedding, then q and the key and value caches
};

/// RMSNorm carried through the products: an operand bf16(h gamma) and, per
/// row of h, its sums of squares over 32 columns each, [m][width / 32]. The
/// rows' factors rsqrt(sum / width + eps) scale the product's outputs.
struct Norm {
  const Bf16* gamma = nullptr;  // [width]
  Bf16* scaled = nullptr;       // [m][width]
  float* squares = nullptr;     // [m][width / 32]
  float eps = 0.0F;
};

/// What QkvRope's launch takes (dit_kernels.hpp); head_dim a multiple of 32.
struct Qkv {
  const float* rope = nullptr;  // [positions][head_dim] cos | sin, or null
  const std::int32_t* positions = nullptr;
  const std::int32_t* cache_rows = nullptr;
  float* q = nullptr;
  float* k_cache = nullptr;
  float* v_cache = nullptr;
  int heads = 0;
  int kv_heads = 0;
  int head_dim = 0;
  int capacity = 0;
};

struct Product {
  const Bf16* x = nullptr;  // [m][k]
  const void* w = nullptr;  // panels: Q8_0 expanded to bf16(scale q), or bf16
  bool bf16 = false;
  std::size_t m = 0;
  std::size_t k = 0;
  std::size_t n = 0;
  Out kind = Out::kStore;
  float* y = nullptr;
  Bf16* out = nullptr;
  Norm norm;  // kSwiGlu, kQkvCache: of x; kAccumulate: of y, made when norm.scaled is set
  Qkv qkv;
};

/// Whether the kernels take the product's sizes (their 32-bit offsets).
bool Supported(std::size_t m, std::size_t k, std::size_t n);

/// Workgroup tile `shape`: rows, columns and k groups.
struct Shape {
  int bm, bn, groups;
};
constexpr int kShapes = 7;
Shape ShapeOf(int shape);
/// The shape an m x k x n product takes, and its modelled time.
int PickShape(std::size_t m, std::size_t k, std::size_t n, double* microseconds = nullptr,
              Out kind = Out::kStore);
/// Whether a standalone product of more than 128 rows takes these kernels
/// (`q8`: Q8_0 panels, else bf16 panels).
bool Use(std::size_t m, std::size_t k, std::size_t n, bool q8);
/// Whether an m x k x n product of Q8_0 panels with the exact per-block
/// arithmetic (33 to 128 rows) takes RunExact rather than the engine.
bool UseExact(std::size_t m, std::size_t k, std::size_t n);
/// The product with each 32-column block's float32 sum scaled into the row's
/// (kernels/wmma_products.hip:192-215): kStore, kAccumulate or kBf16.
int RunExact(const Product& p, hipStream_t stream);
Shape ExactShape();
/// The norm's operand of rows h [m][width], width a multiple of 32.
void Scale(const float* h, const Norm& norm, std::size_t m, std::size_t width,
           hipStream_t stream);
/// Launches the product (arguments checked by the caller: CheckProduct; k a
/// multiple of 32, and n where the norm or SwiGLU take part). A non-negative `shape` forces that one
/// (not the 160-row tiles for kQkvCache).
int Run(const Product& p, hipStream_t stream, int shape = -1);

}  // namespace vx::prefill

#endif  // VOXCPM_AMD_Q8_PREFILL_HPP_
