// Q8_0 (or bf16) panels x bfloat16 rows for more than 128 rows, the
// reference's expansion of Q8_0 weights to bf16(f16 scale * q) with one
// float32 sum over k (gemm.cpp:305-312, kernels/wmma_products.hip:94-112),
// on gfx950's 32 x 32 x 16 bf16 matrix cores.
//
// The panels hold each lane's operand bytes together, so a wave loads its
// columns' weights straight into registers, expands them there and multiplies
// them with every row of the workgroup's tile: only the activations pass
// through LDS. (With both operands in LDS a 64 x 64 wave tile reads 16 KB per
// 16 MFMAs, as much as the LDS delivers in their time.) Four to eight waves
// along n share a tile's rows; where a product has too few tiles for the
// compute units, KG groups of waves take a run of k each and their sums meet
// in LDS in group order, which needs no second launch. k advances 64 columns
// (a panel pair) per step, with two steps' weights and activations in flight
// and one barrier per step.
//
// A wave's 32-column tile is two panel groups of 16 rows: neighbours, or for
// SwiGLU a gate group and its up group, for the rotary embedding a head's two
// halves, whose sums then sit 16 lanes apart. A residual add's epilogue leaves
// the next RMSNorm's operand and each row's sums of squares over 32 columns
// each, which the next product's workgroups add up for their rows' factors: a
// launch less per norm (3 to 5 us, 2 us of them back in the epilogues).
//
// What bounds them: up to about 200 tiles of few steps the launch, the first
// loads and the sums' meeting (4 to 6 us), then about 0.85 us a step, whose
// products take 0.45 us (128 x 256): the rest is the wait for the step's
// barrier and first operands, which two more steps in flight shortened
// (1.0 -> 0.88 us). Measured on MI355X against the tiled, split and
// 64-row-block kernels these replaced (Q8_0, us): 310 x 1024 x 2560 17.1 ->
// 7.9, 310 x 2048 x 1024 8.9 -> 7.4, 310 x 1024 x 8192 17.3 -> 12.1,
// 310 x 4096 x 1024 14.0 -> 10.6, 617 x 2048 x 2560 22.6 -> 13.9, 617 x 6144 x
// 2048 57 -> 28, 617 x 2048 x 12288 64 -> 36, 777 x 2048 x 12288 56 -> 41; bf16
// 333 x 4096 x 1024 15.7 -> 11.7. The matrix cores are busy for 55 % of the 160 x
// 256 tiles' time at 777 x 2048 x 12288, 24 to 36 % in a prompt's products.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "bf16x3.hpp"
#include "common.hpp"
#include "products.hpp"
#include "q8.hpp"
#include "q8_prefill.hpp"
#include "q8_tile.hpp"

namespace vx::prefill {
namespace {

using bf16x3::F32x16;
using q8::AsBf16x8;

constexpr int kDies = 8;

struct Args {
  const Bf16* x;
  const std::uint8_t* w;
  float* y;
  Bf16* out;
  int m, k, n;
  int pairs, groups;
  int m_tiles;
  int tiles;
  int pair_stride;  // panel groups from a column tile's first group to its second
  Norm norm;
  Qkv qkv;
};

/// Workgroup b runs on die b % 8: die d takes a contiguous range of tiles (a
/// weight tile's row tiles first), so that its L2 serves their weights.
__device__ inline int DieOrdered(int b, int blocks) {
  const int per = blocks / kDies;
  const int extra = blocks % kDies;
  const int die = b % kDies;
  return die * per + min(die, extra) + b / kDies;
}

/// LDS index of 16-byte chunk `chunk` (0..7) of 128-byte row `row`: the rows
/// alternate between the halves of a 256-byte bank line, so the chunk swaps
/// with row / 2.
__device__ inline int Swizzled(int row, int chunk) {
  return row * 8 + (chunk ^ ((row >> 1) & 7));
}

/// BM rows, FN 32-column tiles per wave, NW waves along n, KG groups of k,
/// DW steps' weights in flight per wave.
template<int BM, int FN, int NW, int KG, int DW>
struct Tile {
  static constexpr int kFn = FN;
  static constexpr int kNw = NW;
  static constexpr int kKg = KG;
  static constexpr int kDw = DW;
  // Operands a quarter step ahead where the registers allow (up to two waves
  // per SIMD); with four waves per SIMD they cover each other's waits.
  static constexpr bool kAhead = KG <= 2;
  static constexpr int kBm = BM;
  static constexpr int kFm = BM / 32;
  static constexpr int kColumns = 32 * FN * NW;
  static constexpr int kGroupThreads = NW * kWave;
  static constexpr int kThreads = kGroupThreads * KG;
  static constexpr int kPieces = BM * 8 / kGroupThreads;  // 16-byte x pieces per thread per step
  static constexpr int kStageBytes = 2 * BM * 128;        // per group
  // Four groups and more share the sums' meeting: each adds all groups' of
  // its share of the values; of two the first adds the second's.
  static constexpr bool kShared = KG >= 4;
  static constexpr int kMeetBytes = (kShared ? KG : KG - 1) * BM * kColumns * 4;
  // Threads that add a row's sums of squares.
  static constexpr int kRowThreads = kThreads / BM >= 32   ? 32
                                     : kThreads / BM >= 16 ? 16
                                     : kThreads / BM >= 4  ? 4
                                     : kThreads / BM >= 2  ? 2
                                                           : 1;
  static constexpr int kLds = KG * kStageBytes > kMeetBytes ? KG * kStageBytes : kMeetBytes;
};

/// MODE: the weights' arithmetic.
enum Mode : int { kExpanded = 0, kPanels16 = 1, kExact = 2 };

template<class T, int MODE, int OUT>
__global__ __launch_bounds__(T::kThreads, T::kThreads / 256) void PrefillKernel(Args a) {
  constexpr bool BF16 = MODE == kPanels16;
  constexpr bool EXACT = MODE == kExact;
  constexpr int FN = T::kFn;
  constexpr int NW = T::kNw;
  constexpr int KG = T::kKg;
  constexpr int DW = BF16 ? 2 : T::kDw;  // bf16 panels take twice the registers
  constexpr int kUnit = BF16 ? q8::kBf16UnitBytes : q8::kUnitBytes;
  constexpr int kFm = T::kFm;
  constexpr int kPieces = T::kPieces;
  constexpr int kLoads = BF16 ? 4 : 2;  // 16-byte weight loads per column tile and step
  // Vector instructions of a quarter step (expansion of 8 FN weights, about
  // 25 each, and addresses) per product.
  constexpr int kShare = ((BF16 ? 0 : 22) * FN + 8) / (kFm * FN) + 1;
  constexpr bool kNormed = OUT == static_cast<int>(Out::kSwiGlu) ||
                           OUT == static_cast<int>(Out::kQkvCache);
  constexpr bool kPaired = kNormed;  // a column tile's groups lie pair_stride apart
  __shared__ __align__(16) unsigned char lds[T::kLds];
  __shared__ float row_scale[kNormed ? T::kBm : 1];
  constexpr bool kQkv = OUT == static_cast<int>(Out::kQkvCache);
  __shared__ std::int32_t row_position[kQkv ? T::kBm : 1];
  __shared__ std::int32_t row_cache[kQkv ? T::kBm : 1];

  const int lane = static_cast<int>(threadIdx.x) % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int group = wave / NW;  // of k
  const int wn = wave % NW;
  const int tid = static_cast<int>(threadIdx.x) % T::kGroupThreads;
  uint4* const stages = reinterpret_cast<uint4*>(lds) + group * (T::kStageBytes / 16);
  const int tile = DieOrdered(static_cast<int>(blockIdx.x), a.tiles);
  const int row0 = __builtin_amdgcn_readfirstlane((tile % a.m_tiles) * T::kBm);
  const int n_tile = __builtin_amdgcn_readfirstlane(tile / a.m_tiles);
  const int steps = (a.pairs + KG - 1) / KG;
  const int first = group * steps;
  const int last = min(a.pairs, first + steps);

  const __amdgpu_buffer_rsrc_t x_buffer = q8::BufferOf(
      a.x, 2U * static_cast<std::uint32_t>(a.m) * static_cast<std::uint32_t>(a.k));
  // Column tile j: panel groups first_group(j) and pair_stride further on.
  const int column_tile = n_tile * (FN * NW) + wn * FN;
  const auto first_group = [&](int j) {
    const int at = column_tile + j;
    // A rotary tile: 16 dimensions of a head's first half and of its second.
    return OUT == static_cast<int>(Out::kQkvCache)
               ? at / a.pair_stride * 2 * a.pair_stride + at % a.pair_stride
           : OUT == static_cast<int>(Out::kSwiGlu) ? at
                                                   : 2 * at;
  };
  const std::uint32_t group_bytes = static_cast<std::uint32_t>(a.pairs) * kUnit;
  __amdgpu_buffer_rsrc_t w_buffer[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int g = first_group(j);
    const int left = max(0, min(a.groups - g, a.pair_stride + 1));
    w_buffer[j] = q8::BufferOf(a.w + static_cast<std::size_t>(g) * group_bytes,
                               static_cast<std::uint32_t>(left) * group_bytes);
  }
  const std::uint32_t w_lane =
      static_cast<std::uint32_t>(lane % 32 / 16) * static_cast<std::uint32_t>(a.pair_stride) *
          group_bytes +
      16U * static_cast<std::uint32_t>(16 * (lane / 32) + lane % 16);
  const std::uint32_t s_lane =
      static_cast<std::uint32_t>(lane % 32 / 16) * static_cast<std::uint32_t>(a.pair_stride) *
          group_bytes +
      q8::kValueBytes + 4U * static_cast<std::uint32_t>(lane % 16);

  struct Weights {
    uint4 v[FN][kLoads];
    std::uint32_t scales[FN];
  };
  // Load i of a tile: octets 2 i + lane / 32 of both blocks (Q8_0), or of
  // block i / 2 octets 2 (i % 2) + lane / 32 (bf16).
  const auto load_weights = [&](int step, Weights& w) {
    const bool live = step < last;
    const std::uint32_t unit = static_cast<std::uint32_t>(step) * kUnit;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i)
        w.v[j][i] = q8::BufferLoad16(
            w_buffer[j],
            w_lane + unit + (BF16 ? 1024U * (i / 2) + 512U * (i % 2) : 512U * i), live);
      if constexpr (!BF16)
        w.scales[j] = q8::BufferLoad4(w_buffer[j], s_lane + unit, live);
    }
  };
  const auto weights_of = [&](const Weights& w, int j, int block, int half) {
    if constexpr (BF16)
      return AsBf16x8(w.v[j][2 * block + half]);
    const uint4& v = w.v[j][half];
    if constexpr (EXACT)
      return block == 0 ? q8::Int8x8ToBf16(v.x, v.y) : q8::Int8x8ToBf16(v.z, v.w);
    const float scale = HalfValue(static_cast<std::uint16_t>(
        block == 0 ? w.scales[j] & 0xFFFFU : w.scales[j] >> 16));
    return AsBf16x8(block == 0 ? q8::Expand(v.x, v.y, scale) : q8::Expand(v.z, v.w, scale));
  };
  std::uint32_t x_at[kPieces];
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    const int piece = tid + T::kGroupThreads * i;
    const int row = row0 + piece / 8;
    x_at[i] = row < a.m ? 2U * static_cast<std::uint32_t>(row * a.k + 8 * (piece % 8))
                        : q8::kPastBuffer;
  }
  const auto load_x = [&](int step, int i) {
    const int column = 64 * step + 8 * ((tid + T::kGroupThreads * i) % 8);
    return q8::BufferLoad16(x_buffer, x_at[i] + 128U * static_cast<std::uint32_t>(step),
                            step < last && column < a.k && x_at[i] != q8::kPastBuffer);
  };
  const auto store_x = [&](int stage, int i, const uint4& v) {
    const int piece = tid + T::kGroupThreads * i;
    stages[stage * T::kBm * 8 + Swizzled(piece / 8, piece % 8)] = v;
  };

  F32x16 acc[kFm][FN];
#pragma unroll
  for (int i = 0; i < kFm; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        acc[i][j][v] = 0.0F;
  uint4 xs[2][kPieces];
  Weights ws[DW];
  // In the order they are waited for: a wait covers every older load.
#pragma unroll
  for (int i = 0; i < kPieces; ++i)
    xs[0][i] = load_x(first, i);
  load_weights(first, ws[0]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < kPieces; ++i)
    xs[1][i] = load_x(first + 1, i);
#pragma unroll
  for (int d = 1; d < DW; ++d) {
    load_weights(first + d, ws[d]);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    store_x(0, i, xs[0][i]);
    xs[0][i] = load_x(first + 2, i);
  }
  if constexpr (kNormed) {
    const int row = static_cast<int>(threadIdx.x) / T::kRowThreads;
    const int part = static_cast<int>(threadIdx.x) % T::kRowThreads;
    const int count = a.k / 32;
    if (row < T::kBm) {  // whole groups of kRowThreads lanes
      const int from = min(row0 + row, a.m - 1);
      const float* const squares = a.norm.squares + static_cast<std::size_t>(from) * count;
      float sum = 0.0F;
      if (count % 4 == 0) {
        const float4* const quads = reinterpret_cast<const float4*>(squares);
#pragma unroll 8
        for (int i = part; i < count / 4; i += T::kRowThreads)
          sum += quads[i].x + quads[i].y + (quads[i].z + quads[i].w);
      } else {
        for (int i = part; i < count; i += T::kRowThreads)
          sum += squares[i];
      }
      if constexpr (OUT == static_cast<int>(Out::kQkvCache)) {
        if (part == 0) {
          row_position[row] = a.qkv.positions[from];
          row_cache[row] = a.qkv.cache_rows[from];
        }
      }
#pragma unroll
      for (int offset = T::kRowThreads / 2; offset > 0; offset /= 2)
        sum += __shfl_xor(sum, offset, kWave);
      if (part == 0)
        row_scale[row] = rsqrtf(sum / static_cast<float>(a.k) + a.norm.eps);
    }
  }
  const auto multiply = [&](const uint4(&x)[kFm], const q8::Bf16x8(&w)[FN]) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int i = 0; i < kFm; ++i)
        acc[i][j] = bf16x3::Mfma32(AsBf16x8(x[i]), w[j], acc[i][j]);
  };
  // The operands of a step's quarters (16 columns of k). Ahead: two at a
  // time, each quarter read and expanded under the products of the one
  // before it, the first under the last quarter of the step before (of the
  // first step: zeros).
  uint4 x_operand[2][kFm];
  q8::Bf16x8 w_operand[2][FN];
  F32x16 block_sum[EXACT ? kFm : 1];
  if constexpr (T::kAhead) {
#pragma unroll
    for (int i = 0; i < kFm; ++i)
      x_operand[1][i] = uint4{0U, 0U, 0U, 0U};
#pragma unroll
    for (int j = 0; j < FN; ++j)
      w_operand[1][j] = AsBf16x8(uint4{0U, 0U, 0U, 0U});
  }
  __syncthreads();
  for (int step0 = 0; step0 < steps; step0 += DW) {
#pragma unroll
    for (int d = 0; d < DW; ++d) {
      if (step0 + d >= steps)
        break;
      const int step = first + step0 + d;
      // LDS stage d % 2 and weight set d hold the step, the other register
      // set of x the next one.
      const int next = 1 - d % 2;
      const uint4* const rows = stages + d % 2 * T::kBm * 8;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const int now = T::kAhead ? kk % 2 : 0;
#pragma unroll
        for (int i = 0; i < kFm; ++i)
          x_operand[now][i] = rows[Swizzled(32 * i + lane % 32, 2 * kk + lane / 32)];
        if constexpr (T::kAhead)
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < FN; ++j)
          w_operand[now][j] = weights_of(ws[d], j, kk / 2, kk % 2);
        const int ready = T::kAhead ? 1 - now : 0;
        if constexpr (EXACT) {
          // A block's float32 sum from zero, then scaled into the row's.
          static_assert(!EXACT || (!T::kAhead && FN == 1), "exact tiles");
#pragma unroll
          for (int i = 0; i < kFm; ++i) {
            if (kk % 2 == 0) {
#pragma unroll
              for (int v = 0; v < 16; ++v)
                block_sum[i][v] = 0.0F;
            }
            block_sum[i] = bf16x3::Mfma32(AsBf16x8(x_operand[0][i]), w_operand[0][0],
                                          block_sum[i]);
            if (kk % 2 == 1) {
              const float scale = HalfValue(static_cast<std::uint16_t>(
                  kk == 1 ? ws[d].scales[0] & 0xFFFFU : ws[d].scales[0] >> 16));
#pragma unroll
              for (int v = 0; v < 16; ++v)
                acc[i][0][v] = __builtin_fmaf(scale, block_sum[i][v], acc[i][0][v]);
            }
          }
        } else {
          multiply(x_operand[ready], w_operand[ready]);
        }
#pragma unroll
        for (int i = kk * kPieces / 4; i < (kk + 1) * kPieces / 4; ++i) {
          store_x(next, i, xs[next][i]);
          xs[next][i] = load_x(step + 3, i);
        }
        if (kk == 3)
          load_weights(step + DW, ws[d]);
        if constexpr (T::kAhead) {
          // A share of the vector instructions behind every product.
#pragma unroll
          for (int q = 0; q < kFm * FN; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, kShare, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __syncthreads();
    }
  }
  if constexpr (T::kAhead)
    multiply(x_operand[1], w_operand[1]);
  if constexpr (KG > 1)
    __syncthreads();  // the stages have been read: the sums take their place

  // The tile's output rows as one buffer: rows past m lie past it, and its
  // range check drops them. Element e of column tile j: row 32 (e / 16) +
  // 8 (e % 16 / 4) + 4 (lane / 32) + e % 4 of the tile, column lane % 32.
  constexpr bool kSwiGlu = OUT == static_cast<int>(Out::kSwiGlu);
  constexpr std::uint32_t kBytes = kSwiGlu || OUT == static_cast<int>(Out::kBf16) ? 2 : 4;
  const std::uint32_t width = static_cast<std::uint32_t>(kSwiGlu ? a.n / 2 : a.n);
  const std::uint32_t row_bytes = width * kBytes;
  const __amdgpu_buffer_rsrc_t out = q8::BufferOf(
      (kBytes == 2 ? reinterpret_cast<unsigned char*>(a.out)
                   : reinterpret_cast<unsigned char*>(a.y)) +
          static_cast<std::size_t>(row0) * row_bytes,
      static_cast<std::uint32_t>(min(T::kBm, a.m - row0)) * row_bytes);
  const auto row_of = [&](int at) {
    return 32 * (at / 16) + 8 * (at % 16 / 4) + 4 * (lane / 32) + at % 4;
  };
  // This lane's and its pair's value of a paired tile: lanes 0-15 of each 32
  // hold the first group, the lane 16 on the second.
  const auto pair_of = [&](float value) {
    const auto swapped = __builtin_amdgcn_permlane16_swap(
        __float_as_uint(value), __float_as_uint(value), false, false);
    return __uint_as_float(lane % 32 < 16 ? swapped[1] : swapped[0]);
  };
  // The rotary factors of elements e0 .. of column tile j: 1 and 0 where
  // nothing rotates.
  const auto load_rotary = [&](auto count, float* c, float* s, int e0, int j) {
    constexpr int kCount = decltype(count)::value;
    const int at = column_tile + j;
    const bool rotates = a.qkv.rope != nullptr &&
                         at / a.pair_stride < a.qkv.heads + a.qkv.kv_heads;
#pragma unroll
    for (int e = 0; e < kCount; ++e) {
      c[e] = 1.0F;
      s[e] = 0.0F;
      if (rotates) {
        const float* const table =
            a.qkv.rope +
            static_cast<std::size_t>(row_position[row_of(e0 + e)]) * a.qkv.head_dim +
            16 * (at % a.pair_stride) + lane % 16;
        c[e] = table[0];
        s[e] = table[a.qkv.head_dim / 2];
      }
    }
  };
  const auto emit_qkv = [&](auto count, const float* value, const float* c, const float* s,
                            int e0, int j) {
    constexpr int kCount = decltype(count)::value;
    const Qkv& o = a.qkv;
    const int at = column_tile + j;
    const int head = at / a.pair_stride;
    if (32 * at >= a.n)
      return;
    const bool second = lane % 32 >= 16;
    const int dim = 16 * (at % a.pair_stride) + lane % 16 + (second ? o.head_dim / 2 : 0);
    const bool rotates = o.rope != nullptr && head < o.heads + o.kv_heads;
    // Query heads lie [row][head], a cache's [row] of its head.
    const bool query = head < o.heads;
    float* const base =
        query ? o.q + static_cast<std::size_t>(head) * o.head_dim + dim
              : (head < o.heads + o.kv_heads ? o.k_cache : o.v_cache) +
                    static_cast<std::size_t>((head - o.heads) % o.kv_heads) * o.capacity *
                        o.head_dim +
                    dim;
    const std::size_t stride = static_cast<std::size_t>(query ? o.heads : 1) * o.head_dim;
#pragma unroll
    for (int e = 0; e < kCount; ++e) {
      const int local = row_of(e0 + e);
      const float own = value[e] * row_scale[local];
      const float other = pair_of(own);
      const float rotated = !rotates ? own
                            : second ? own * c[e] + other * s[e]
                                     : own * c[e] - other * s[e];
      if (row0 + local < a.m)
        base[static_cast<std::size_t>(query ? row0 + local : row_cache[local]) * stride] = rotated;
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const auto emit = [&](auto count, const float* value, int e0, int j) {
    constexpr int kCount = decltype(count)::value;
    if constexpr (kQkv) {
      float c[kCount], s[kCount];
      load_rotary(count, c, s, e0, j);
      emit_qkv(count, value, c, s, e0, j);
      return;
    }
    const std::uint32_t column = static_cast<std::uint32_t>(
        kSwiGlu ? 16 * (column_tile + j) + lane % 16 : 32 * (column_tile + j) + lane % 32);
    const bool writes = column < width && (!kSwiGlu || lane % 32 < 16);
    int offset[kCount];
#pragma unroll
    for (int e = 0; e < kCount; ++e) {
      const int row = row_of(e0 + e);
      offset[e] = static_cast<int>(
          writes ? static_cast<std::uint32_t>(row) * row_bytes + kBytes * column
                 : q8::kPastBuffer);
    }
    if constexpr (kSwiGlu) {
#pragma unroll
      for (int e = 0; e < kCount; ++e) {
        const float gate = value[e] * row_scale[row_of(e0 + e)];
        const float up = pair_of(gate);
        __builtin_amdgcn_raw_buffer_store_b16(
            q8::Bf16Fast(gate / (1.0F + expf(-gate)) * up), out, offset[e], 0, 0);
      }
    } else if constexpr (OUT == static_cast<int>(Out::kBf16)) {
#pragma unroll
      for (int e = 0; e < kCount; ++e)
        __builtin_amdgcn_raw_buffer_store_b16(q8::Bf16Fast(value[e]), out, offset[e], 0, 0);
    } else {
      float prior[kCount];
#pragma unroll
      for (int e = 0; e < kCount; ++e)
        prior[e] = OUT == static_cast<int>(Out::kAccumulate)
                       ? __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                       out, offset[e], 0, 0))
                       : 0.0F;
#pragma unroll
      for (int e = 0; e < kCount; ++e) {
        const float sum =
            OUT == static_cast<int>(Out::kAccumulate) ? prior[e] + value[e] : value[e];
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(std::uint32_t, sum), out,
                                              offset[e], 0, 0);
        prior[e] = sum;
      }
      if (OUT == static_cast<int>(Out::kAccumulate) && a.norm.scaled != nullptr) {
        // The next norm's operand and this column tile's sums of squares.
        const float gamma = writes ? Bf16Value(a.norm.gamma[column]) : 0.0F;
#pragma unroll
        for (int e = 0; e < kCount; ++e) {
          const int row = row0 + row_of(e0 + e);
          const float square = AddXor16(RowSum16(writes ? prior[e] * prior[e] : 0.0F));
          if (row >= a.m || !writes)
            continue;
          a.norm.scaled[static_cast<std::size_t>(row) * width + column] =
              q8::Bf16Fast(prior[e] * gamma);
          if (lane % 32 == 0)
            a.norm.squares[static_cast<std::size_t>(row) * (width / 32) + column_tile + j] =
                square;
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // one tile's values at a time
  };
  constexpr int kValues = kFm * FN * 16;
  float* const sums = reinterpret_cast<float*>(lds);  // [groups][values][group threads]
  const auto put = [&](int slot) {
#pragma unroll
    for (int i = 0; i < kFm; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const float element = acc[i][j][v];
          sums[(slot * kValues + (i * FN + j) * 16 + v) * T::kGroupThreads + tid] = element;
        }
  };
  if constexpr (T::kShared) {
    static_assert(FN == 1, "a share lies within one column tile");
    constexpr int kShare = kValues / KG;
    const std::integral_constant<int, kShare> share;
    float c[kShare], s[kShare];  // loaded while the sums meet
    if constexpr (kQkv)
      load_rotary(share, c, s, group * kShare, 0);
    put(group);
    __syncthreads();
    float value[kShare];
#pragma unroll
    for (int e = 0; e < kShare; ++e)
      value[e] = sums[(group * kShare + e) * T::kGroupThreads + tid];
#pragma unroll
    for (int g = 1; g < KG; ++g)
#pragma unroll
      for (int e = 0; e < kShare; ++e)
        value[e] += sums[(g * kValues + group * kShare + e) * T::kGroupThreads + tid];
    if constexpr (kQkv)
      emit_qkv(share, value, c, s, group * kShare, 0);
    else
      emit(share, value, group * kShare, 0);
    return;
  }
  if constexpr (KG == 2) {
    if (group == 1)
      put(0);
    __syncthreads();
    if (group == 1)
      return;
  }
#pragma unroll
  for (int i = 0; i < kFm; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      float value[16];
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        value[v] = acc[i][j][v];
        if constexpr (KG == 2)
          value[v] += sums[((i * FN + j) * 16 + v) * T::kGroupThreads + tid];
      }
      emit(std::integral_constant<int, 16>{}, value, 16 * i, j);
    }
}

/// One thread per four columns: bf16(h gamma), and the sums of squares of
/// eight threads' 32 columns.
__global__ void ScaleKernel(const float* h, Norm norm, int m, int width) {
  const std::size_t at =
      (static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x) * 4;
  if (at >= static_cast<std::size_t>(m) * width)  // whole groups of eight lanes
    return;
  const int column = static_cast<int>(at % static_cast<std::size_t>(width));
  const float4 x = *reinterpret_cast<const float4*>(h + at);
  const ushort4 gamma = *reinterpret_cast<const ushort4*>(norm.gamma + column);
  *reinterpret_cast<uint2*>(norm.scaled + at) =
      uint2{q8::PackBf16x2(x.x * Bf16Value(gamma.x), x.y * Bf16Value(gamma.y)),
            q8::PackBf16x2(x.z * Bf16Value(gamma.z), x.w * Bf16Value(gamma.w))};
  float square = x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w;
#pragma unroll
  for (int offset = 4; offset > 0; offset /= 2)
    square += __shfl_xor(square, offset, kWave);
  if (threadIdx.x % 8 == 0)
    norm.squares[at / 32] = square;
}

/// The caches' epilogue over 160-row tiles does not unroll (its sums would
/// lie in memory): PickShape leaves them out.
constexpr int kNoQkvRows = 160;
template<class T>
constexpr bool kTakesQkv = T::kBm != kNoQkvRows;

template<class T>
void Launch(const Product& p, Args a, hipStream_t stream) {
  a.m_tiles = static_cast<int>((p.m + T::kBm - 1) / T::kBm);
  a.tiles = a.m_tiles * static_cast<int>((p.n + T::kColumns - 1) / T::kColumns);
  const auto launch = [&](auto kernel) { kernel<<<a.tiles, T::kThreads, 0, stream>>>(a); };
  if (p.bf16) {
    switch (p.kind) {
      case Out::kStore: launch(PrefillKernel<T, kPanels16, 0>); break;
      case Out::kAccumulate: launch(PrefillKernel<T, kPanels16, 1>); break;
      case Out::kBf16: launch(PrefillKernel<T, kPanels16, 2>); break;
      case Out::kSwiGlu: launch(PrefillKernel<T, kPanels16, 3>); break;
      case Out::kQkvCache:
        if constexpr (kTakesQkv<T>)
          launch(PrefillKernel<T, kPanels16, 4>);
        break;
    }
  } else {
    switch (p.kind) {
      case Out::kStore: launch(PrefillKernel<T, kExpanded, 0>); break;
      case Out::kAccumulate: launch(PrefillKernel<T, kExpanded, 1>); break;
      case Out::kBf16: launch(PrefillKernel<T, kExpanded, 2>); break;
      case Out::kSwiGlu: launch(PrefillKernel<T, kExpanded, 3>); break;
      case Out::kQkvCache:
        if constexpr (kTakesQkv<T>)
          launch(PrefillKernel<T, kExpanded, 4>);
        break;
    }
  }
}

/// The exact kernels' one tile: 32 x 32, sixteen groups of k. Each 32-column
/// block's products sum from zero on the matrix cores and are then scaled
/// into the group's sums (kernels/wmma_products.hip:192-215).
using ExactTile = Tile<32, 1, 1, 16, 2>;

}  // namespace

namespace {

/// A shape and its model in microseconds, one workgroup per compute unit: each
/// round of workgroups takes `fixed` and `step` per step (64 columns of k of a
/// group), and a full grid's tiles share another `share` per step (memory and
/// L2). Fitted on MI355X to 14700 times of both weight formats, forced to each
/// shape (m 129..3000, k 64..6144, n 64..24576): the picked shape took on average
/// 0.3 % longer than the best one, one time in twenty over 2 % longer, and the
/// times lie within a sixth of the model's nine times in ten, long outputs of
/// short reductions apart.
struct Model {
  Shape shape;
  double fixed, step, share;
};
constexpr Model kModels[kShapes] = {
    {{128, 256, 1}, 5.9, 0.58, 0.49}, {{128, 128, 2}, 5.2, 0.60, 0.53},
    {{64, 128, 4}, 5.3, 0.86, 0.37},  {{64, 64, 8}, 5.5, 1.12, 0.26},
    {{32, 64, 8}, 4.0, 0.84, 0.09},   {{160, 256, 1}, 6.5, 0.66, 0.61},
    {{96, 256, 1}, 5.1, 0.53, 0.35}};
constexpr std::size_t kComputeUnits = 256;

double Time(const Model& model, std::size_t m, std::size_t k, std::size_t n) {
  const std::size_t groups = static_cast<std::size_t>(model.shape.groups);
  const std::size_t tiles =
      ((m + model.shape.bm - 1) / model.shape.bm) * ((n + model.shape.bn - 1) / model.shape.bn);
  const double rounds = static_cast<double>((tiles + kComputeUnits - 1) / kComputeUnits);
  const double steps = static_cast<double>((q8::Pairs(k) + groups - 1) / groups);
  return rounds * (model.fixed + steps * model.step) +
         static_cast<double>(tiles) / kComputeUnits * steps * model.share;
}

}  // namespace

Shape ShapeOf(int shape) { return kModels[shape].shape; }

Shape ExactShape() { return Shape{ExactTile::kBm, ExactTile::kColumns, ExactTile::kKg}; }

bool Supported(std::size_t m, std::size_t k, std::size_t n) {
  // The output tile, the activations and a column tile's panels as buffers
  // of 32-bit offsets.
  return n <= (std::size_t{1} << 20) && m * k <= (std::size_t{1} << 29) &&
         q8::Bf16PackedBytes(n, k) < (std::size_t{1} << 31);
}

int PickShape(std::size_t m, std::size_t k, std::size_t n, double* microseconds, Out kind) {
  int best = 0;
  double least = 0.0;
  for (int i = 0; i < kShapes; ++i) {
    if (kind == Out::kQkvCache && kModels[i].shape.bm == kNoQkvRows)
      continue;
    const double time = Time(kModels[i], m, k, n);
    if (i == 0 || time < least) {
      best = i;
      least = time;
    }
  }
  if (microseconds != nullptr)
    *microseconds = least;
  return best;
}

bool Use(std::size_t m, std::size_t k, std::size_t n, bool q8) {
  // Q8_0 products of up to 512 rows over 6144 columns of k and more stay on the
  // kernels whose split over k uses a scratch: a caller's, or the static one of
  // the entry that cannot allocate, whose use at 300 and 320 x 6144 x 2048 the
  // tests hold fast. These kernels would be the faster ones there too (300 x
  // 6144 x 2048 31.6 us there, 20.7 here; 129 x 18.1 and 14.7; 512 x 6144 x 4096
  // 59.3 and 35.6). bf16 panels have no such entry, and the stacks, which use no
  // scratch, come here.
  if (m <= kExactRows || !Supported(m, k, n) || (q8 && k >= 6144 && m <= 512))
    return false;
  // Else by both sides' times in microseconds, fitted on MI355X (drawn and
  // gridded sizes, both weight formats, replayed from a graph).
  double here = 0.0;
  PickShape(m, k, n, &here);
  const double pairs = static_cast<double>(q8::Pairs(k));
  if (UseRowBlocks(m, k, n, q8)) {
    // 2936 sizes, m 129..1500, k 64..6144, n 64..16384: on average 0.6 %
    // slower than the faster kernel, one in fifty over 4 % slower than in row
    // blocks. 129 x 256 x 1024 3.7 us there, 6.4 here; 256 x 1024 x 1024 4.8 and
    // 6.0; 512 x 544 x 2055 12.5 and 8.9; 448 x 1536 x 2560 16.4 and 11.5.
    const double output = static_cast<double>(m) * static_cast<double>(n) * 1e-6;  // its writing
    const std::size_t blocks = (m + 63) / 64;
    const std::size_t groups = q8::Groups(n);
    const std::size_t wide = groups <= 256 ? 1 : 2;  // row groups per workgroup
    const std::size_t tiles = (groups + wide - 1) / wide;
    const double rounds =
        static_cast<double>((blocks * tiles + kComputeUnits - 1) / kComputeUnits * wide);
    const double passes = static_cast<double>((q8::Pairs(k) + 15) / 16);  // of 16 waves
    // A tile's blocks share a die, and its L2, where tiles are whole eights.
    const double pair = tiles % kDies == 0 ? 0.064 : 0.079;
    // The workgroups' rounds, or the rows' reading by few tiles.
    const double there =
        std::max(2.7 + 0.41 * passes + rounds * (0.21 + pair * pairs) + 2.5 * output,
                 2.7 + 0.0083 * static_cast<double>(blocks) * pairs);
    return here + 0.3 * output < there;
  }
  if (!UseGemm(m, n))  // the tiled kernel, slower wherever it was measured
    return true;
  // 962 sizes, m 384..3000, k 64..6144, n 6144..24576: on average 0.7 % slower
  // than the faster kernel, one in 35 over 4 % slower than the 256-row tiles. bf16
  // 1024 x 2048 x 12288 56 us there, 64 here; 777 x 2048 x 12288 56 and 41.
  const GemmPlan plan = PlanGemm(m, k, n, 0);
  const Model gemm = plan.bn == 256 ? Model{{256, 256, 1}, 10.9, 0.83, 1.08}
                                    : Model{{256, 128, 1}, 7.1, 0.48, 0.59};
  return here < Time(gemm, m, k, n);
}

void Scale(const float* h, const Norm& norm, std::size_t m, std::size_t width,
           hipStream_t stream) {
  const std::size_t quads = m * width / 4;
  ScaleKernel<<<static_cast<unsigned>((quads + 255) / 256), 256, 0, stream>>>(
      h, norm, static_cast<int>(m), static_cast<int>(width));
}

namespace {

Args ArgsOf(const Product& p) {
  Args a{};
  a.x = p.x;
  a.w = static_cast<const std::uint8_t*>(p.w);
  a.y = p.y;
  a.out = p.out;
  a.m = static_cast<int>(p.m);
  a.k = static_cast<int>(p.k);
  a.n = static_cast<int>(p.n);
  a.pairs = static_cast<int>(q8::Pairs(p.k));
  a.groups = static_cast<int>(q8::Groups(p.n));
  a.pair_stride = p.kind == Out::kSwiGlu      ? a.groups / 2
                  : p.kind == Out::kQkvCache ? p.qkv.head_dim / 32
                                             : 1;
  a.norm = p.norm;
  a.qkv = p.qkv;
  return a;
}

}  // namespace

bool UseExact(std::size_t m, std::size_t k, std::size_t n) {
  // Past 64 rows the engine needs a second block of rows, and past 32 rows over
  // more than 128 row groups a second round of workgroups, each of which reads
  // all of its block's x: over more than 4096 columns of k these tiles are faster
  // there while they take one round (77 x 6144 x 2055 19.1 -> 11.5 us, 128 x 8192 x
  // 2048 18.4 -> 14.5, 65 x 5120 x 130 10.3 -> 9.6, 77 x 4128 x 2048 10.4 -> 10.2, 33 x
  // 6144 x 2049 12.5 -> 10.7, 64 x 5120 x 4096 15.5 -> 10.9 on MI355X). Below, the
  // engine is (64 x 6144 x 2048 10.3 there, 11.0 here; 48 x 8192 x 1024 10.8 and
  // 12.1; 32 x 6144 x 4000 9.6 and 11.8). Over shorter k its sums come out
  // closer to 64 bits (100 x 1024 x 1024 7.0e-8 there, 8.3e-8 here; 77 x 6144 x 2048
  // 1.06e-7 and 1.01e-7, 40 x 4128 x 2560 9.4e-8 and 9.2e-8).
  return (m > 64 || (m > 32 && n > 2048)) && m <= kExactRows && k > 4096 &&
         Supported(m, k, n) && ((m + 31) / 32) * ((n + 31) / 32) <= kComputeUnits;
}

int RunExact(const Product& p, hipStream_t stream) {
  Args a = ArgsOf(p);
  a.m_tiles = static_cast<int>((p.m + 31) / 32);
  a.tiles = a.m_tiles * static_cast<int>((p.n + 31) / 32);
  const auto launch = [&](auto kernel) {
    kernel<<<a.tiles, ExactTile::kThreads, 0, stream>>>(a);
  };
  if (p.kind == Out::kBf16)
    launch(PrefillKernel<ExactTile, kExact, 2>);
  else if (p.kind == Out::kAccumulate)
    launch(PrefillKernel<ExactTile, kExact, 1>);
  else
    launch(PrefillKernel<ExactTile, kExact, 0>);
  return LaunchStatus("exact product");
}

int Run(const Product& p, hipStream_t stream, int shape) {
  const Args a = ArgsOf(p);
  if (shape < 0)
    shape = PickShape(p.m, p.k, p.n, nullptr, p.kind);
  switch (shape) {
    case 0: Launch<Tile<128, 2, 4, 1, 4>>(p, a, stream); break;
    case 1: Launch<Tile<128, 1, 4, 2, 4>>(p, a, stream); break;
    case 2: Launch<Tile<64, 1, 4, 4, 2>>(p, a, stream); break;
    case 3: Launch<Tile<64, 1, 2, 8, 2>>(p, a, stream); break;
    case 4: Launch<Tile<32, 1, 2, 8, 2>>(p, a, stream); break;
    case 5: Launch<Tile<160, 2, 4, 1, 4>>(p, a, stream); break;
    default: Launch<Tile<96, 2, 4, 1, 4>>(p, a, stream); break;
  }
  return LaunchStatus("prefill product");
}

}  // namespace vx::prefill
