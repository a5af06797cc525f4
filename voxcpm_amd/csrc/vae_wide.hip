// The AudioVAE decoder over many rows (vae.cpp:415-502 of the reference):
// its products on gfx950's f16 matrix cores with float32 operands split into
// two float16 terms (f16x2.hpp: three products of a sixteenth of the float32
// instructions' time each), and a residual unit as one launch at 32 and 64
// channels.
//
// ProductKernel computes BM x BN tiles of y = A W^T with four waves, k in
// steps of 32: two steps' float32 operands are in flight in registers, and
// while a step is multiplied from LDS the next one is split into the other
// LDS buffer (two planes of 64-byte rows, 16-byte chunk c of row r at
// c ^ ((r / 4) % 4)), one barrier per step.
//
// UnitKernel computes all C channels of about 128 rows, 32 input channels
// at a time: the stream's rows with the 6 d before them pass through Snake
// into LDS once, a thread makes four outputs d rows apart of the depthwise
// convolution from ten of them (28 reads otherwise), passes them through
// the second Snake, splits them into the operand planes, and the waves
// multiply with the split weights. The stream is read and written once per
// unit (its rows before the tile's by two workgroups), where a launch per
// step moved it six times: units of the shallow blocks are bound by that
// traffic. In and out are two buffers: a tile's history rows belong to the
// tile before it.
//
// A workgroup that has met operands outside the float16 pairs' range (kLeast,
// 65504) starts over from three bfloat16 terms (bf16x3.hpp), which span
// float32's: nothing is stored before its last product, and the histories it
// leaves are the same values again.
//
// Measured on MI355X over 125 frames at VoxCPM2's shape, per launch, against
// the float32 kernels' (F32TileKernel and a depthwise launch per unit):
// transposed convolutions 112 / 132 / 176 / 110 / 72 / 52 -> 51 / 57 / 62 /
// 36 / 25 / 30 us; units of 1024 / 512 / 256 / 128 channels 36 / 60 / 106 /
// 83 -> 26 / 34 / 43 / 40 us, of 64 and 32 (fused) 87 / 82 -> 28 / 23 us; the
// decode 2090 -> 820-875 us on several cards, its error against 64 bits 4.6e-5 ->
// 1.7e-5. The 128 x 128 products keep the matrix cores busy for 14 % (units of
// 128 channels) to 45 % (block 1's transposed convolution) of their time and the
// vector unit, which splits the operands, for 33 to 48 %; the fused units wait
// on memory (61 MB in 23 us; vector unit 45 to 62 %). Units of 128 channels measured
// the same fused as in two launches, of 256 slower.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "bf16x3.hpp"
#include "common.hpp"
#include "f16x2.hpp"
#include "q8.hpp"
#include "q8_tile.hpp"
#include "snake.hpp"
#include "vae_wide.hpp"

namespace vx::vae {
namespace {

using bf16x3::F32x16;
using f16x2::Octet;

constexpr int kThreads = 256;
constexpr int kTaps = 7;
constexpr int kStep = 32;  // reduction columns per step
constexpr int kDies = 8;
// Eight neighbouring operands of a row (four, of a unit's activations) are to
// hold a magnitude of at least this, or zeros alone: the pairs' absolute error
// of 2^-36 is then at most 2^-21 of their largest. (Weights of spread 0.001
// and activations of spread 0.05 hold such a group once in 10^13.)
constexpr float kLeast = 0x1p-15F;

/// 16-byte chunk `chunk` (8 values of 16 bits) of row `row` of a plane of 64-byte
/// rows: the equal chunks of 16 consecutive rows (a 16-lane group of a
/// 16-byte read) fall on distinct banks.
__device__ inline int PlaneIndex(int row, int chunk) {
  return row * 4 + (chunk ^ ((row >> 2) & 3));
}

__device__ inline float4 Load4(__amdgpu_buffer_rsrc_t buffer, std::uint32_t offset, bool keep) {
  return __builtin_bit_cast(float4, q8::BufferLoad16(buffer, offset, keep));
}

/// Two planes of a split operand: 32 columns of ROWS rows.
template<int ROWS>
struct Planes {
  uint4 data[2][ROWS * 4];
  __device__ void Store(int row, int chunk, const uint4& first, const uint4& second) {
    const int at = PlaneIndex(row, chunk);
    data[0][at] = first;
    data[1][at] = second;
  }
  __device__ Octet Load(int row, int chunk) const {
    const int at = PlaneIndex(row, chunk);
    return Octet{data[0][at], data[1][at]};
  }
};

/// The history rows of a target, copied by one workgroup.
__device__ inline void CopyHistory(const Epilogue& e, int n) {
  const int count = e.target == Target::kBlockInput ? n
                    : e.target == Target::kOutput   ? (kTaps - 1) * n
                                                    : 0;
  for (int i = static_cast<int>(threadIdx.x); i < count; i += static_cast<int>(blockDim.x))
    e.out[i] = e.history[i];
}

/// Stores one wave's 32 x 32 accumulator tile at (row0, column0): rows below
/// `row_end` (at most the product's `t`), `n` columns in all. The buffers end
/// at row_end, whose range check drops the rows past it.
__device__ inline void StoreTile(const Epilogue& e, const F32x16& acc, int row0, int column0,
                                 int row_end, int t, int n) {
  const int lane = static_cast<int>(threadIdx.x) % kWave;
  const int column = column0 + lane % 32;
  if (column >= n)
    return;
  const float bias = e.bias[e.channels == n ? column : column % e.channels];
  SnakeChannel snake;
  float scale = 1.0F;
  float shift = 0.0F;
  if (e.target != Target::kStream)
    snake = SnakeChannel(e.alpha[column]);
  if (e.target == Target::kBlockInput) {
    scale = e.scale[column];
    shift = e.shift[column];
  }
  const int row1 = row0 + 4 * (lane / 32);
  const std::uint32_t row_bytes = 4U * static_cast<std::uint32_t>(n);
  const std::uint32_t first = static_cast<std::uint32_t>(row1) * row_bytes +
                              4U * static_cast<std::uint32_t>(column);
  const auto offset = [&](int v) {
    return static_cast<int>(first + static_cast<std::uint32_t>(8 * (v / 4) + v % 4) * row_bytes);
  };
  const int before = e.target == Target::kBlockInput ? 1
                     : e.target == Target::kOutput   ? kTaps - 1
                                                     : 0;
  const std::uint32_t bytes = static_cast<std::uint32_t>(row_end) * row_bytes;
  const __amdgpu_buffer_rsrc_t out =
      q8::BufferOf(e.out + static_cast<std::size_t>(before) * n, bytes);
  F32x16 value = acc;
  if (e.prior != nullptr) {
    const __amdgpu_buffer_rsrc_t priors = q8::BufferOf(e.prior, bytes);
    F32x16 prior;
#pragma unroll
    for (int v = 0; v < 16; ++v)
      prior[v] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(priors, offset(v), 0, 0));
    value = prior + acc;
  }
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    float x = value[v] + bias;
    if (e.target == Target::kBlockInput)
      x = snake(x * scale + shift);
    else if (e.target == Target::kOutput)
      x = snake(x);
    value[v] = x;
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(std::uint32_t, x), out, offset(v), 0,
                                          0);
  }
  if (e.target == Target::kBlockInput && row_end == t && row0 + 32 >= t) {
#pragma unroll
    for (int v = 0; v < 16; ++v)
      if (row1 + 8 * (v / 4) + v % 4 == t - 1)
        e.history_next[column] = value[v];
  }
  // One tile's values at a time.
  __builtin_amdgcn_sched_barrier(0);
}

// ---- products ------------------------------------------------------------------

struct ProductArgs {
  Product p;
  int m_tiles;
  int n_tiles;
  int columns_first;  // consecutive tiles of a die share weights (else rows)
};

/// Workgroup b runs on die b % 8: die d takes a contiguous range of tiles,
/// so that neighbouring tiles share its L2.
__device__ inline int DieOrdered(int b, int blocks) {
  const int per = blocks / kDies;
  const int extra = blocks % kDies;
  const int die = b % kDies;
  return die * per + min(die, extra) + b / kDies;
}

/// The six kept products of two bfloat16 triples (bf16x3.hpp), from two
/// planes at a time: pass 0 holds h and m, pass 1 h and l.
template<int PASS>
__device__ inline F32x16 MultiplyLarge(const Octet& x, const Octet& w, F32x16 sum) {
  using q8::AsBf16x8;
  sum = bf16x3::Mfma32(AsBf16x8(x.l), AsBf16x8(w.h), sum);
  sum = bf16x3::Mfma32(AsBf16x8(x.h), AsBf16x8(w.l), sum);
  if constexpr (PASS == 0) {
    sum = bf16x3::Mfma32(AsBf16x8(x.l), AsBf16x8(w.l), sum);
    sum = bf16x3::Mfma32(AsBf16x8(x.h), AsBf16x8(w.h), sum);
  }
  return sum;
}

/// A workgroup's tile of the product and what its threads hold of it. KG
/// groups of four waves take a run of k each; their sums meet in LDS in
/// group order.
template<int BM, int BN, int KG>
struct ProductTile {
  static constexpr int kFm = BM / 64;  // 32 x 32 tiles of a wave (waves 2 x 2)
  static constexpr int kFn = BN / 64;
  static constexpr int kPiecesA = BM * 4 / kThreads;  // pieces of eight values per thread
  static constexpr int kPieces = kPiecesA + BN * 4 / kThreads;
  using Sums = F32x16[kFm][kFn];
  struct Stages {
    Planes<BM> a[2];
    Planes<BN> b[2];
  };
  struct Shared {
    Stages stages[KG];
    int restart;
  };
  static_assert((KG - 1) * sizeof(float) * BM * BN <= KG * sizeof(Stages), "the groups' sums");

  const Product& p;
  Shared& shared;
  Stages& own;  // the group's
  int row0, column0;
  int first, last, steps;  // the group's steps: `steps` from first, none from `last` on
  int lane, group, wm, wn, chunk, piece_row;
  __amdgpu_buffer_rsrc_t x_buffer, w_buffer;
  std::uint32_t at[kPieces];

  __device__ ProductTile(const ProductArgs& a, Shared& s)
      : p(a.p), shared(s),
        own(s.stages[__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kThreads)]) {
    const int tid = static_cast<int>(threadIdx.x) % kThreads;
    lane = tid % kWave;
    group = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kThreads);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    wm = wave / 2;
    wn = wave % 2;
    const int tiles = a.m_tiles * a.n_tiles;
    const int tile = DieOrdered(static_cast<int>(blockIdx.x), tiles);
    const int m_tile = a.columns_first != 0 ? tile % a.m_tiles : tile / a.n_tiles;
    const int n_tile = a.columns_first != 0 ? tile / a.m_tiles : tile % a.n_tiles;
    row0 = __builtin_amdgcn_readfirstlane(m_tile * BM);
    column0 = __builtin_amdgcn_readfirstlane(n_tile * BN);
    steps = (p.k / kStep + KG - 1) / KG;
    first = group * steps;
    last = min(p.k / kStep, first + steps);
    // With taps, A's row f is u(f) | u(f - 1), rows of k / 2 at x from u(-1).
    const int stride = p.taps ? p.k / 2 : p.k;
    x_buffer = q8::BufferOf(p.x, 4U * static_cast<std::uint32_t>(p.taps ? p.t + 1 : p.t) *
                                     static_cast<std::uint32_t>(stride));
    w_buffer =
        q8::BufferOf(p.w, 4U * static_cast<std::uint32_t>(p.n) * static_cast<std::uint32_t>(p.k));
    // Piece i of a thread: chunk tid % 4 of A's row tid / 4 + 64 i, or of
    // W's from piece kPiecesA on.
    chunk = tid % 4;
    piece_row = tid / 4;
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int row = i < kPiecesA ? row0 + piece_row + 64 * i
                                   : column0 + piece_row + 64 * (i - kPiecesA);
      const bool live = row < (i < kPiecesA ? p.t : p.n);
      const int from = i < kPiecesA ? (row + (p.taps ? 1 : 0)) * stride : row * p.k;
      at[i] = live ? 4U * static_cast<std::uint32_t>(from + 8 * chunk) : q8::kPastBuffer;
    }
  }

  __device__ void Load(int step, int i, float4 (&v)[2]) const {
    const int column = step * kStep;
    // u(f - 1)'s column c of the second half sits a row before u(f)'s.
    const std::uint32_t offset = 4U * static_cast<std::uint32_t>(
                                          i < kPiecesA && p.taps && column >= p.k / 2
                                              ? column - p.k
                                              : column);
    const bool keep = step < last && at[i] != q8::kPastBuffer;
    if (i < kPiecesA) {
      v[0] = Load4(x_buffer, at[i] + offset, keep);
      v[1] = Load4(x_buffer, at[i] + offset + 16U, keep);
    } else {
      v[0] = Load4(w_buffer, at[i] + offset, keep);
      v[1] = Load4(w_buffer, at[i] + offset + 16U, keep);
    }
  }
  __device__ void Store(int stage, int i, const uint4& h, const uint4& l) const {
    if (i < kPiecesA)
      own.a[stage].Store(piece_row + 64 * i, chunk, h, l);
    else
      own.b[stage].Store(piece_row + 64 * (i - kPiecesA), chunk, h, l);
  }
  /// The operands of reduction half s (16 columns) of a stage.
  __device__ void Read(int stage, int s, Octet (&x)[kFm], Octet (&w)[kFn]) const {
#pragma unroll
    for (int i = 0; i < kFm; ++i)
      x[i] = own.a[stage].Load((BM / 2) * wm + 32 * i + lane % 32, 2 * s + lane / 32);
#pragma unroll
    for (int j = 0; j < kFn; ++j)
      w[j] = own.b[stage].Load((BN / 2) * wn + 32 * j + lane % 32, 2 * s + lane / 32);
  }
  __device__ static void Clear(Sums& sums) {
#pragma unroll
    for (int i = 0; i < kFm; ++i)
#pragma unroll
      for (int j = 0; j < kFn; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          sums[i][j][v] = 0.0F;
  }

  /// The tile from float16 pairs; false (in every thread) when operands
  /// lie outside their range.
  template<int SETS>
  __device__ bool Multiply(Sums& acc) {
    float4 values[SETS][kPieces][2];  // steps in flight
    Sums cross;                       // hl + lh, 2048 times their value
    Clear(acc);
    Clear(cross);
    f16x2::Range range;
    const auto split_piece = [&](int stage, int i, const float4 (&v)[2]) {
      const Octet o = f16x2::Split(v[0], v[1]);
      Store(stage, i, o.h, o.l);
      range.Add(f16x2::Largest(f16x2::Largest(0.0F, v[0]), v[1]));
    };
#pragma unroll
    for (int set = 0; set < SETS; ++set)
#pragma unroll
      for (int i = 0; i < kPieces; ++i)
        Load(first + set, i, values[set][i]);
    if (threadIdx.x == 0)
      shared.restart = 0;
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      split_piece(0, i, values[0][i]);
      Load(first + SETS, i, values[0][i]);
    }
    __syncthreads();
    for (int step0 = first; step0 < first + steps; step0 += 2) {
#pragma unroll
      for (int stage = 0; stage < 2; ++stage) {
        const int step = step0 + stage;
        if (step >= first + steps)
          break;
        // LDS stage `stage` holds the step, the register set the next one.
        float4(&next)[kPieces][2] = values[SETS == 1 ? 0 : 1 - stage];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          Octet x[kFm], w[kFn];
          Read(stage, s, x, w);
#pragma unroll
          for (int i = 0; i < kFm; ++i)
#pragma unroll
            for (int j = 0; j < kFn; ++j)
              cross[i][j] = f16x2::Mfma32(x[i].l, w[j].h, cross[i][j]);
#pragma unroll
          for (int i = 0; i < kFm; ++i)
#pragma unroll
            for (int j = 0; j < kFn; ++j)
              acc[i][j] = f16x2::Mfma32(x[i].h, w[j].h, acc[i][j]);
#pragma unroll
          for (int i = 0; i < kFm; ++i)
#pragma unroll
            for (int j = 0; j < kFn; ++j)
              cross[i][j] = f16x2::Mfma32(x[i].h, w[j].l, cross[i][j]);
#pragma unroll
          for (int i = s * kPieces / 2; i < (s + 1) * kPieces / 2; ++i) {
            split_piece(1 - stage, i, next[i]);
            Load(step + 1 + SETS, i, next[i]);
          }
        }
        __syncthreads();
      }
    }
    if (!range.Holds(kLeast))
      shared.restart = 1;
#pragma unroll
    for (int i = 0; i < kFm; ++i)
#pragma unroll
      for (int j = 0; j < kFn; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[i][j][v] = __builtin_fmaf(cross[i][j][v], f16x2::kCross, acc[i][j][v]);
    __syncthreads();
    return shared.restart == 0;
  }

  /// The tile from bfloat16 triples.
  __device__ void MultiplyFullRange(Sums& acc) {
    Clear(acc);
#pragma unroll 1
    for (int step = first; step < first + steps; ++step) {
      float4 values[kPieces][2];
#pragma unroll
      for (int i = 0; i < kPieces; ++i)
        Load(step, i, values[i]);
      const auto pass = [&](auto index) {
        constexpr int kPass = decltype(index)::value;
        __syncthreads();  // the planes have been read
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
          const bf16x3::Octet o = bf16x3::Split(values[i][0], values[i][1]);
          Store(0, i, o.h, kPass == 0 ? o.m : o.l);
        }
        __syncthreads();
#pragma unroll 1
        for (int s = 0; s < 2; ++s) {
          Octet x[kFm], w[kFn];
          Read(0, s, x, w);
#pragma unroll
          for (int i = 0; i < kFm; ++i)
#pragma unroll
            for (int j = 0; j < kFn; ++j)
              acc[i][j] = MultiplyLarge<kPass>(x[i], w[j], acc[i][j]);
        }
      };
      pass(std::integral_constant<int, 0>{});
      pass(std::integral_constant<int, 1>{});
    }
  }

  /// Adds the other groups' sums to the first's.
  __device__ void Meet(Sums& acc) const {
    float* const sums = reinterpret_cast<float*>(shared.stages);  // [KG - 1][values][kThreads]
    constexpr int kValues = kFm * kFn * 16;
    const int tid = static_cast<int>(threadIdx.x) % kThreads;
    __syncthreads();  // the stages have been read
    if (group > 0) {
#pragma unroll
      for (int e = 0; e < kValues; ++e)
        sums[((group - 1) * kValues + e) * kThreads + tid] =
            acc[e / 16 / kFn][e / 16 % kFn][e % 16];
    }
    __syncthreads();
    if (group > 0)
      return;
#pragma unroll
    for (int g = 0; g < KG - 1; ++g)
#pragma unroll
      for (int e = 0; e < kValues; ++e)
        acc[e / 16 / kFn][e / 16 % kFn][e % 16] += sums[(g * kValues + e) * kThreads + tid];
  }

  __device__ void Finish(const Sums& acc) const {
    const int row = row0 + (BM / 2) * wm;
    const int column = column0 + (BN / 2) * wn;
#pragma unroll
    for (int i = 0; i < kFm; ++i)
#pragma unroll
      for (int j = 0; j < kFn; ++j)
        StoreTile(p.epilogue, acc[i][j], row + 32 * i, column + 32 * j, p.t, p.t, p.n);
  }
};

template<int BM, int BN, int KG>
__global__ __launch_bounds__(kThreads * KG, KG == 1 ? 2 : KG) void ProductKernel(ProductArgs a) {
  using Tile = ProductTile<BM, BN, KG>;
  __shared__ typename Tile::Shared shared;
  const Product& p = a.p;
  if (blockIdx.x == 0) {
    CopyHistory(p.epilogue, p.n);
    if (p.tail != nullptr)
      for (int i = static_cast<int>(threadIdx.x); i < p.k / 2; i += kThreads * KG)
        p.tail[i] = p.x[static_cast<std::size_t>(p.t - 1) * p.k + i];
  }
  Tile tile(a, shared);
  typename Tile::Sums acc;
  if (!tile.template Multiply<BM == 128 ? 1 : 2>(acc))
    tile.MultiplyFullRange(acc);
  if constexpr (KG > 1) {
    tile.Meet(acc);
    if (tile.group > 0)
      return;
  }
  tile.Finish(acc);
}

// ---- residual units ------------------------------------------------------------

constexpr int kUnitRows = 128;                      // rows of a workgroup's MFMA tiles
/// Rows a workgroup computes: whole runs of four rows d apart, so that every
/// item of four outputs is one thread's.
__host__ __device__ constexpr int RowsOf(int d) { return kUnitRows / (4 * d) * (4 * d); }

struct UnitArgs {
  Unit u;
  const float* w;
  Epilogue epilogue;
};

/// The 28 taps, bias and Snake constants of a quad of channels.
struct QuadTaps {
  float4 w[kTaps];  // channel s's tap j is flat element 7 s + j
  float4 bias;
  float4 alpha;
  __device__ void Load(const Unit& u, int channel) {
    const float4* from = reinterpret_cast<const float4*>(u.taps + channel * kTaps);
#pragma unroll
    for (int i = 0; i < kTaps; ++i)
      w[i] = from[i];
    bias = *reinterpret_cast<const float4*>(u.bias + channel);
    alpha = *reinterpret_cast<const float4*>(u.alpha_out + channel);
  }
  __device__ float Tap(int s, int j) const {
    const int flat = kTaps * s + j;
    const float4& v = w[flat / 4];
    return flat % 4 == 0 ? v.x : flat % 4 == 1 ? v.y : flat % 4 == 2 ? v.z : v.w;
  }
};

/// Snake of a quad of channels.
struct Snake4 {
  SnakeChannel x, y, z, w;
  __device__ explicit Snake4(const float4& a) : x(a.x), y(a.y), z(a.z), w(a.w) {}
  __device__ float4 operator()(const float4& v) const {
    return make_float4(x(v.x), y(v.y), z(v.z), w(v.w));
  }
};

/// Snake(bias + sum_j tap_j rows[i + j]) of outputs i = 0 .. 3, the taps in
/// order.
__device__ inline void Convolve(const QuadTaps& taps, const float4 (&rows)[10], float4 (&out)[4]) {
  const Snake4 snake(taps.alpha);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float4 sum = taps.bias;
#pragma unroll
    for (int j = 0; j < kTaps; ++j) {
      sum.x += taps.Tap(0, j) * rows[i + j].x;
      sum.y += taps.Tap(1, j) * rows[i + j].y;
      sum.z += taps.Tap(2, j) * rows[i + j].z;
      sum.w += taps.Tap(3, j) * rows[i + j].w;
    }
    out[i] = snake(sum);
  }
}

template<int C, int D>
struct UnitTile {
  static constexpr int kTiles = C / 32;  // output column tiles
  static constexpr int kHalo = (kTaps - 1) * D;
  static constexpr int kRows = RowsOf(D);
  static constexpr int kWindowRows = kRows + kHalo;
  static constexpr int kLoads = (kWindowRows * 8 + kThreads - 1) / kThreads;
  // Pieces of eight weights per thread.
  static constexpr int kPieces = (C * 4 + kThreads - 1) / kThreads;
  using Sums = F32x16[kTiles];
  struct Shared {
    Planes<kUnitRows> a;
    Planes<C> w;
    float4 window[kWindowRows * 8];  // [rows][8]
    int restart;
  };

  const Unit& u;
  Shared& shared;
  int lane, wave, row0;
  int quad;      // channels 4 quad .. + 3 of every step
  int slot0;     // window slot i: row slot0 + 32 i (the stream's row0 - 6 d + that)
  bool live;     // this thread's item: outputs item_row + i d, i = 0 .. 3, of its quad
  int item_row;
  __amdgpu_buffer_rsrc_t w_buffer;
  __amdgpu_buffer_rsrc_t y_buffer;

  __device__ UnitTile(const UnitArgs& a, Shared& s) : u(a.u), shared(s) {
    const int tid = static_cast<int>(threadIdx.x);
    lane = tid % kWave;
    wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    row0 = static_cast<int>(blockIdx.x) * kRows;
    quad = tid % 8;
    slot0 = tid / 8;
    live = slot0 < kRows / 4;
    item_row = live ? slot0 % D + 4 * (slot0 / D) * D : 0;
    w_buffer = q8::BufferOf(a.w, 4U * C * C);
    y_buffer = q8::BufferOf(u.y, 4U * C * static_cast<std::uint32_t>(u.t));
  }

  /// Rows past the stream's end read zero (they reach no output row).
  __device__ void LoadWindow(int channel, float4 (&ys)[kLoads]) const {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int slot = slot0 + 32 * i;
      const int row = row0 - kHalo + slot;
      ys[i] = Load4(y_buffer, 4U * static_cast<std::uint32_t>(row * C + channel + 4 * quad),
                    row >= 0 && slot < kWindowRows);
    }
    if (blockIdx.x != 0)
      return;
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      if (slot0 + 32 * i < kHalo)
        ys[i] = *reinterpret_cast<const float4*>(u.state + (slot0 + 32 * i) * C + channel +
                                                 4 * quad);
  }
  /// Snake of the loaded rows into the window, and the chunk's last rows
  /// into the next chunk's history.
  __device__ void StoreWindow(int channel, const float4 (&ys)[kLoads]) const {
    const int c = channel + 4 * quad;
    const Snake4 snake(*reinterpret_cast<const float4*>(u.alpha_in + c));
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int slot = slot0 + 32 * i;
      const int row = row0 - kHalo + slot;
      if (slot >= kWindowRows)
        continue;
      const float4 v = row < 0 ? ys[i] : snake(ys[i]);
      shared.window[slot * 8 + quad] = v;
      if (slot >= kHalo && row >= u.t - kHalo && row < u.t)
        *reinterpret_cast<float4*>(u.state_next +
                                   static_cast<std::size_t>(row - (u.t - kHalo)) * C + c) = v;
    }
  }
  __device__ void Item(const QuadTaps& taps, float4 (&out)[4]) const {
    float4 in[10];
#pragma unroll
    for (int l = 0; l < 10; ++l)
      in[l] = shared.window[(item_row + l * D) * 8 + quad];
    Convolve(taps, in, out);
  }
  __device__ void StoreItem(int i, const uint2& first, const uint2& second) const {
    const int at = 2 * PlaneIndex(item_row + i * D, quad / 2) + quad % 2;
    reinterpret_cast<uint2*>(shared.a.data[0])[at] = first;
    reinterpret_cast<uint2*>(shared.a.data[1])[at] = second;
  }
  __device__ void LoadWeights(int channel, int piece, float4 (&v)[2]) const {
    const std::uint32_t at =
        4U * static_cast<std::uint32_t>((piece / 4) * C + channel + 8 * (piece % 4));
    v[0] = Load4(w_buffer, at, piece < 4 * C);
    v[1] = Load4(w_buffer, at + 16U, piece < 4 * C);
  }
  __device__ Octet ReadX(int s) const {
    return shared.a.Load(32 * wave + lane % 32, 2 * s + lane / 32);
  }
  __device__ Octet ReadW(int j, int s) const {
    return shared.w.Load(32 * j + lane % 32, 2 * s + lane / 32);
  }
  __device__ static void Clear(Sums& acc) {
#pragma unroll
    for (int j = 0; j < kTiles; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        acc[j][v] = 0.0F;
  }

  /// The unit's product from float16 pairs; false (in every thread) when an
  /// operand passed their range.
  __device__ bool Multiply(Sums& acc) const {
    const int tid = static_cast<int>(threadIdx.x);
    float4 ys[kLoads];
    float4 ws[kPieces][2];
    f16x2::Range range;
    Clear(acc);
    if (tid == 0)
      shared.restart = 0;
    LoadWindow(0, ys);
#pragma unroll
    for (int i = 0; i < kPieces; ++i)
      LoadWeights(0, tid + kThreads * i, ws[i]);
#pragma unroll
    for (int channel = 0; channel < C; channel += kStep) {
      __syncthreads();  // the step before has been multiplied
      StoreWindow(channel, ys);
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        const int piece = tid + kThreads * i;
        const Octet o = f16x2::Split(ws[i][0], ws[i][1]);
        if (piece < 4 * C)
          shared.w.Store(piece / 4, piece % 4, o.h, o.l);
        range.Add(f16x2::Largest(f16x2::Largest(0.0F, ws[i][0]), ws[i][1]));
      }
      __syncthreads();
      if (channel + kStep < C) {
        LoadWindow(channel + kStep, ys);
#pragma unroll
        for (int i = 0; i < kPieces; ++i)
          LoadWeights(channel + kStep, tid + kThreads * i, ws[i]);
      }
      if (live) {
        QuadTaps taps;
        taps.Load(u, channel + 4 * quad);
        float4 out[4];
        Item(taps, out);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f16x2::Pair p0 = f16x2::Split(out[i].x, out[i].y);
          const f16x2::Pair p1 = f16x2::Split(out[i].z, out[i].w);
          StoreItem(i, uint2{p0.h, p1.h}, uint2{p0.l, p1.l});
          range.Add(f16x2::Largest(0.0F, out[i]));
        }
      }
      __syncthreads();
      const Octet x0 = ReadX(0);
      const Octet x1 = ReadX(1);
#pragma unroll
      for (int j = 0; j < kTiles; ++j) {
        const Octet w0 = ReadW(j, 0);
        const Octet w1 = ReadW(j, 1);
        F32x16 cross;
#pragma unroll
        for (int v = 0; v < 16; ++v)
          cross[v] = 0.0F;
        cross = f16x2::Mfma32(x0.l, w0.h, cross);
        acc[j] = f16x2::Mfma32(x0.h, w0.h, acc[j]);
        cross = f16x2::Mfma32(x0.h, w0.l, cross);
        acc[j] = f16x2::Mfma32(x1.h, w1.h, acc[j]);
        cross = f16x2::Mfma32(x1.l, w1.h, cross);
        cross = f16x2::Mfma32(x1.h, w1.l, cross);
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[j][v] = __builtin_fmaf(cross[v], f16x2::kCross, acc[j][v]);
        // Two tiles' operands and cross terms in registers at a time.
        if (j % 2 == 1)
          __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (!range.Holds(kLeast))
      shared.restart = 1;
    __syncthreads();
    return shared.restart == 0;
  }

  /// The unit's product from bfloat16 triples.
  __device__ void MultiplyFullRange(Sums& acc) const {
    Clear(acc);
#pragma unroll 1
    for (int channel = 0; channel < C; channel += kStep) {
      float4 ys[kLoads];
      LoadWindow(channel, ys);
      __syncthreads();
      StoreWindow(channel, ys);
      __syncthreads();
      float4 out[4];
      QuadTaps taps;
      taps.Load(u, channel + 4 * quad);
      Item(taps, out);
      const auto pass = [&](auto index) {
        constexpr int kPass = decltype(index)::value;
        __syncthreads();  // the planes have been read
        if (live) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const bf16x3::Pair p0 = bf16x3::Split(out[i].x, out[i].y);
            const bf16x3::Pair p1 = bf16x3::Split(out[i].z, out[i].w);
            StoreItem(i, uint2{p0.h, p1.h}, kPass == 0 ? uint2{p0.m, p1.m} : uint2{p0.l, p1.l});
          }
        }
#pragma unroll 1
        for (int piece = static_cast<int>(threadIdx.x); piece < 4 * C; piece += kThreads) {
          float4 v[2];
          LoadWeights(channel, piece, v);
          const bf16x3::Octet o = bf16x3::Split(v[0], v[1]);
          shared.w.Store(piece / 4, piece % 4, o.h, kPass == 0 ? o.m : o.l);
        }
        __syncthreads();
#pragma unroll 1
        for (int s = 0; s < 2; ++s) {
          const Octet x = ReadX(s);
#pragma unroll
          for (int j = 0; j < kTiles; ++j)
            acc[j] = MultiplyLarge<kPass>(x, ReadW(j, s), acc[j]);
        }
      };
      pass(std::integral_constant<int, 0>{});
      pass(std::integral_constant<int, 1>{});
    }
  }
};

template<int C, int D>
__global__ __launch_bounds__(kThreads, 3) void UnitKernel(UnitArgs a) {
  using Tile = UnitTile<C, D>;
  __shared__ typename Tile::Shared shared;
  if (blockIdx.x == 0)
    CopyHistory(a.epilogue, C);
  const Tile tile(a, shared);
  typename Tile::Sums acc;
  if (!tile.Multiply(acc))
    tile.MultiplyFullRange(acc);
#pragma unroll
  for (int j = 0; j < Tile::kTiles; ++j)
    StoreTile(a.epilogue, acc[j], tile.row0 + 32 * tile.wave, 32 * j,
              min(tile.row0 + Tile::kRows, a.u.t), a.u.t, C);
}

template<int C>
void LaunchUnit(const UnitArgs& a, hipStream_t stream) {
  const int rows = RowsOf(a.u.d);
  const unsigned grid = static_cast<unsigned>((a.u.t + rows - 1) / rows);
  if (a.u.d == 1)
    UnitKernel<C, 1><<<grid, kThreads, 0, stream>>>(a);
  else if (a.u.d == 3)
    UnitKernel<C, 3><<<grid, kThreads, 0, stream>>>(a);
  else
    UnitKernel<C, 9><<<grid, kThreads, 0, stream>>>(a);
}

/// A thread per quad of channels and four outputs d rows apart.
__global__ __launch_bounds__(kThreads) void DepthwiseWideKernel(Unit u, float* out) {
  const int quads = u.c / 4;
  const int item = static_cast<int>(blockIdx.x) * kThreads + static_cast<int>(threadIdx.x);
  const int task = item / quads;
  const int d = u.d;
  const int halo = (kTaps - 1) * d;
  const int first = task % d + 4 * (task / d) * d;
  if (first >= u.t)
    return;
  const int c = 4 * (item % quads);
  QuadTaps taps;
  taps.Load(u, c);
  const Snake4 snake(*reinterpret_cast<const float4*>(u.alpha_in + c));
  float4 in[10];
#pragma unroll
  for (int l = 0; l < 10; ++l) {
    const int row = first + l * d - halo;
    in[l] = *reinterpret_cast<const float4*>(
        (row < 0 ? u.state + static_cast<std::ptrdiff_t>(row + halo) * u.c
                 : u.y + static_cast<std::ptrdiff_t>(min(row, u.t - 1)) * u.c) +
        c);
  }
#pragma unroll
  for (int l = 0; l < 10; ++l) {
    const int row = first + l * d - halo;
    if (row >= 0)
      in[l] = snake(in[l]);
    if (l >= kTaps - 1 && row >= u.t - halo && row < u.t)
      *reinterpret_cast<float4*>(u.state_next +
                                 static_cast<std::size_t>(row - (u.t - halo)) * u.c + c) = in[l];
  }
  float4 values[4];
  Convolve(taps, in, values);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = first + i * d;
    if (row < u.t)
      *reinterpret_cast<float4*>(out + static_cast<std::size_t>(row) * u.c + c) = values[i];
  }
}

}  // namespace

void RunProduct(const Product& p, hipStream_t stream) {
  const auto tiles = [&](int m, int n) {
    return static_cast<unsigned>(((p.t + m - 1) / m) * ((p.n + n - 1) / n));
  };
  const auto args = [&](int m, int n) {
    // A die re-reads the operand that its tiles do not share: the smaller.
    return ProductArgs{p, (p.t + m - 1) / m, (p.n + n - 1) / n, p.n >= p.t ? 1 : 0};
  };
  // 128 x 128 tiles, k in two groups of waves while they are fewer than one and a
  // half for each compute unit; 64 x 64 with four groups where even two would
  // leave half of the units idle. Lower lines are faster and less exact (a
  // group's sums are the shorter the more groups): with 256 and 128 tiles 72
  // frames decode in 647 us on MI355X instead of 736, 96 in 708 instead of 824, 40
  // in 493 instead of 574 (16, 64 and 125 the same), with an error against 64 bits
  // of 1.79e-5 instead of 1.69e-5 at 96.
  const unsigned big = tiles(128, 128);
  if (big >= 384)
    ProductKernel<128, 128, 1><<<big, kThreads, 0, stream>>>(args(128, 128));
  else if (big >= 180)
    ProductKernel<128, 128, 2><<<big, 2 * kThreads, 0, stream>>>(args(128, 128));
  else
    ProductKernel<64, 64, 4><<<tiles(64, 64), 4 * kThreads, 0, stream>>>(args(64, 64));
}

void RunDepthwise(const Unit& u, float* out, hipStream_t stream) {
  const std::size_t runs = static_cast<std::size_t>((u.t + 4 * u.d - 1) / (4 * u.d));
  const std::size_t items = runs * u.d * (u.c / 4);
  DepthwiseWideKernel<<<static_cast<unsigned>((items + kThreads - 1) / kThreads), kThreads, 0,
                        stream>>>(u, out);
}

bool UnitSupported(std::size_t c) { return c == 32 || c == 64; }

void RunUnit(const Unit& u, const float* w, const Epilogue& epilogue, hipStream_t stream) {
  const UnitArgs a{u, w, epilogue};
  if (u.c == 32)
    LaunchUnit<32>(a, stream);
  else
    LaunchUnit<64>(a, stream);
}

}  // namespace vx::vae
