// The many-row attention over a key/value cache (tile_attention.hip).
#ifndef VOXCPM_AMD_TILE_ATTENTION_HPP_
#define VOXCPM_AMD_TILE_ATTENTION_HPP_

#include <hip/hip_runtime.h>

#include <cstddef>

#include "common.hpp"

namespace vx {

/// Attention's arguments (kernels/generator_kernels.hip:160-241): q
/// [rows][heads][head_dim] rotated and unscaled, one layer's caches
/// [kv_heads][capacity][head_dim], out [rows][heads head_dim] row-major.
struct AttentionShape {
  std::size_t rows, rows_per_sequence, keys_per_sequence, past;
  bool causal;
  std::size_t heads, kv_heads, head_dim, capacity;
};

/// How the matrix-core attention cuts a call's keys.
struct TileAttentionPlan {
  std::size_t chunk = 0;       // keys per chunk
  std::size_t splits = 1;      // chunks of the rows that attend to the most keys
  std::size_t workgroups = 0;  // of the first launch
};

/// Whether the matrix-core attention takes these pointers and this shape,
/// and how.
bool PlanTileAttention(const AttentionShape& s, const float* q, const float* k_cache,
                       const float* v_cache, const Bf16* out, const float* partials,
                       TileAttentionPlan* plan);

/// Whether it is the faster kernel for them: not the split kernel, whose
/// workgroups each take one of `splits` chunks of a row's keys and
/// `heads_per_workgroup` of its heads.
bool UseTileAttention(const AttentionShape& s, const TileAttentionPlan& plan, int splits,
                      int heads_per_workgroup);

/// `partials`: rows x heads x ceil(keys / 64) x (head_dim + 2) floats, or
/// null where a row attends to at most 64 keys.
void TileAttention(const AttentionShape& s, const TileAttentionPlan& plan, const float* q,
                   const float* k_cache, const float* v_cache, Bf16* out, float* partials,
                   hipStream_t stream);

}  // namespace vx

#endif  // VOXCPM_AMD_TILE_ATTENTION_HPP_
