// Products of more than 128 activation rows whose weights go from their
// panels straight into the matrix cores' operands (q8_prefill.hip): the
// stacks' prefill products with their consumers' work in the epilogue, and
// the larger standalone ones.
#ifndef VOXCPM_AMD_Q8_PREFILL_HPP_
#define VOXCPM_AMD_Q8_PREFILL_HPP_

#include <hip/hip_runtime.h>

#include <cstddef>

#include "common.hpp"

namespace vx::prefill {

enum class Out : int {
  kStore = 0,       // y = product
  kAccumulate = 1,  // y += product
  kBf16 = 2,        // out = bf16(product)
  kSwiGlu = 3       // out [m][n / 2] = bf16(silu(gate) up), n / 2 columns each
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
int PickShape(std::size_t m, std::size_t k, std::size_t n, double* microseconds = nullptr);
/// Whether the standalone products of more than 128 rows take these kernels.
bool Use(std::size_t m, std::size_t k, std::size_t n);
/// Launches the product (arguments checked by the caller: CheckProduct; for
/// kSwiGlu n a multiple of 32). A non-negative `shape` forces that one.
int Run(const Product& p, hipStream_t stream, int shape = -1);

}  // namespace vx::prefill

#endif  // VOXCPM_AMD_Q8_PREFILL_HPP_
