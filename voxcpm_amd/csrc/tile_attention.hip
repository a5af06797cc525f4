// Attention of many rows over a float32 key/value cache (a prompt's prefill,
// a prompt's patches through the local encoder): the reference's Attention
// (kernels/generator_kernels.hip:160-241) on gfx950's f16 matrix cores with
// float32 operands split into two float16 terms (f16x2.hpp).
//
// A workgroup of four waves takes 128 queries of one KV head -- a query is a
// (row, query head of the group) pair, so a group's heads share every key
// and value the workgroup brings in -- and a run of keys, 32 at a time:
// the threads load the next 32 keys and values into registers, split the
// current ones into LDS (keys row-major, values transposed), and each wave
// multiplies them with its 32 queries, which stay split in registers.
// Scores are made transposed, S^T = K Q^T, so that a lane holds one query's
// scores (column L % 32) and the exponentials are the next product's B
// operand where they are: O^T = V^T P^T over the keys in the order S^T left
// them, which the transposed values in LDS follow. The softmax runs online
// per query (running maximum and sum, float32).
//
// Short of workgroups, the keys are cut into chunks that separate workgroups
// take, as many as run at once; each leaves its maximum, sum and
// unnormalised values, and a second launch merges a row's chunks in chunk
// order.
//
// A workgroup that met values too small for float16 pairs (kLeast), or whose
// sums came out NaN or infinite, starts over key by key in float32: a value
// past float16's range makes them NaN, and so does a masked key's NaN or
// infinity, whose weight is 0.
//
// Measured on MI355X: 300 rows of 16 heads over 1800 keys 390 us on the
// float32 split kernel, 55 us from three bfloat16 terms (twice the products,
// and 570 workgroups in two rounds), 34.5 us now, of which the merge 7 us. A
// step of one workgroup alone takes 2.1 us, of which the products are 0.65:
// one wave per SIMD runs scores, softmax and values one after the other, and
// registers (230 of 256) leave two workgroups per compute unit. Over the launch
// the matrix cores are busy for 22 % of the time, the vector unit for 47 %.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "bf16x3.hpp"
#include "common.hpp"
#include "f16x2.hpp"
#include "q8.hpp"
#include "q8_tile.hpp"
#include "tile_attention.hpp"

namespace vx {
namespace {

using bf16x3::F32x16;
using f16x2::Octet;

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kQueries = 32 * kWaves;  // per workgroup
constexpr int kKeys = 32;              // per step
// Fewest keys of a chunk (the caller's partials hold a chunk per 64 keys).
constexpr int kLeastChunk = 128;
// Workgroups that run at once, two per compute unit: chunks are cut for as
// many and no more (570 took two rounds; 300 rows over 1800 keys: 384 and 256
// workgroups 44 and 43 us against 43, 700 over 2300 80 and 89 against 71 us).
constexpr std::size_t kTargetWorkgroups = 512;
// A transposed value row in LDS: 32 f16 keys and 16 bytes of padding, so
// that the 16-byte reads of eight consecutive rows fall on distinct banks.
constexpr int kValueRow = 80;
// Eight neighbouring dimensions of a query or a key, four of a value, and one
// dimension of four neighbouring values (of a run's whole quads of keys: the
// fifth key of a five-row patch alone would often fail) are each to hold a
// magnitude of at least this, or zeros alone: the pairs' absolute error of 2^-36 is then 2^-20
// of it, an eight-hundredth of the bfloat16 output's rounding. (Four values
// of spread 0.01 are all smaller once in 5 10^11, of spread 0.001 once in 5 10^7.)
constexpr float kLeast = 0x1p-16F;

struct TileArgs {
  const float* q;
  const float* k;
  const float* v;
  Bf16* out;
  float* values;  // [rows][heads][splits][D], several chunks
  float* stats;   // [rows][heads][splits][2]: maximum, sum
  int rows_per_sequence;
  int keys_per_sequence;
  int past;
  int causal;
  int heads;
  int kv_heads;
  int capacity;
  int sequences;
  int blocks;  // query blocks per (sequence, KV head)
  int chunk;   // keys per chunk
  int splits;  // chunks
  float scale;
};

/// exp(x) for x <= 0 to about one ulp: 2^(x log2 e) with the rounding of
/// the product carried into the result.
__device__ inline float ExpNegative(float x) {
  constexpr float kLog2E = 1.44269504088896341F;
  constexpr float kLog2ELow = 1.92596299e-8F;  // log2 e - kLog2E
  constexpr float kLn2 = 0.693147180559945309F;
  const float a = x * kLog2E;
  const float low = __builtin_fmaf(x, kLog2E, -a) + x * kLog2ELow;
  const float e = __builtin_amdgcn_exp2f(a);
  return __builtin_fmaf(e, low * kLn2, e);
}

/// max over the wave's halves (both lanes of a pair receive it).
__device__ inline float MaxXor32(float x) {
  const auto swapped =
      __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(swapped[0]), __uint_as_float(swapped[1]));
}

/// Most keys of a query of query block `block`.
__device__ inline int BlockKeys(const TileArgs& a, int block, int queries, int group) {
  const int last = min((block + 1) * kQueries, queries) - 1;
  return a.past + (a.causal != 0 ? last / group + 1 : a.rows_per_sequence);
}

template<int D>
__global__ __launch_bounds__(kThreads, 2) void TileAttentionKernel(TileArgs a) {
  constexpr int kChunks = D / 8;    // 16-byte chunks of a key row's plane
  // A key row in LDS: a chunk of padding puts the 16-byte reads of 16
  // consecutive keys on distinct banks.
  constexpr int kKeyRow = kChunks + 1;
  constexpr int kSteps = D / 16;    // MFMA steps of a score
  constexpr int kTiles = D / 32;    // 32-dimension tiles of the output
  constexpr int kKeyLoads = kKeys * kChunks / kThreads;  // 8-value pieces per thread
  constexpr int kValueThreads = kKeys / 4 * (D / 4);     // 4 x 4 pieces
  __shared__ uint4 key_planes[2][kKeys * kKeyRow];
  __shared__ __align__(16) unsigned char value_planes[2][D * kValueRow];
  __shared__ int restart;

  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int column = lane % 32;
  const int half = lane / 32;
  // The grid holds the runs that have keys: sequences and KV heads fastest,
  // then a query block's chunks, the last query blocks, with the most keys
  // of a causal call, first.
  const int heads = a.kv_heads * a.sequences;
  const int g = static_cast<int>(blockIdx.x) % heads % a.kv_heads;
  const int sequence = static_cast<int>(blockIdx.x) % heads / a.kv_heads;
  const int group = a.heads / a.kv_heads;
  const int queries = a.rows_per_sequence * group;
  int split = static_cast<int>(blockIdx.x) / heads;
  int query_block = a.blocks - 1;
  if (a.splits == 1) {
    query_block -= split;
    split = 0;
  } else {
    for (;; --query_block) {
      const int runs = (BlockKeys(a, query_block, queries, group) + a.chunk - 1) / a.chunk;
      if (split < runs)
        break;
      split -= runs;
    }
  }

  // Keys of query `index` (queries past the last count none).
  const auto keys_of = [&](int index) {
    return index >= queries ? 0
                            : a.past + (a.causal != 0 ? index / group + 1 : a.rows_per_sequence);
  };
  const int first_query = query_block * kQueries;
  const int key_begin = split * a.chunk;
  const int key_end =
      min(key_begin + a.chunk, BlockKeys(a, query_block, queries, group));
  const int wave_query = first_query + 32 * wave;
  const int wave_keys =
      wave_query < queries ? keys_of(min(wave_query + 32, queries) - 1) : 0;
  const int query = wave_query + column;
  const int my_keys = keys_of(query);
  // Steps whose keys every query of the wave counts need no mask.
  const int whole_keys = wave_query + 32 <= queries ? keys_of(wave_query) : 0;
  // (row, head) of query `index`, row-major over [rows][heads] (queries past
  // the last take its).
  const auto place = [&](int index) {
    const int local = min(index, queries - 1);
    return (sequence * a.rows_per_sequence + local / group) * a.heads + g * group + local % group;
  };

  // The caches up to the run's end as buffers: loads past it read zero (the
  // cache beyond what was written may hold anything).
  const std::size_t cache = (static_cast<std::size_t>(g) * a.capacity +
                             static_cast<std::size_t>(sequence) * a.keys_per_sequence) *
                            D;
  const std::uint32_t cache_bytes = 4U * D * static_cast<std::uint32_t>(key_end);
  const __amdgpu_buffer_rsrc_t keys = q8::BufferOf(a.k + cache, cache_bytes);
  const __amdgpu_buffer_rsrc_t values = q8::BufferOf(a.v + cache, cache_bytes);
  const auto load16 = [](__amdgpu_buffer_rsrc_t buffer, std::uint32_t offset) {
    return __builtin_bit_cast(float4, q8::BufferLoad16(buffer, offset, true));
  };

  // The next step's keys (pieces of eight values) and values (four keys by
  // four dimensions) in flight.
  float4 key_next[kKeyLoads][2];
  float4 value_next[4];
  const int value_quad = tid % (kKeys / 4);  // keys 4 value_quad .. + 3
  const int dim_quad = tid / (kKeys / 4);    // dimensions 4 dim_quad .. + 3
  const auto load = [&](int key0) {
    const std::uint32_t from = 4U * D * static_cast<std::uint32_t>(key0);
#pragma unroll
    for (int i = 0; i < kKeyLoads; ++i) {
      const std::uint32_t piece = static_cast<std::uint32_t>(tid + kThreads * i);
      key_next[i][0] = load16(keys, from + 32U * piece);
      key_next[i][1] = load16(keys, from + 32U * piece + 16U);
    }
    if (kValueThreads == kThreads || tid < kValueThreads) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        value_next[j] =
            load16(values, from + 4U * static_cast<std::uint32_t>(D * (4 * value_quad + j) +
                                                                  4 * dim_quad));
    }
  };
  f16x2::Least least;  // of what this thread has split
  const auto store = [&](int key0) {
#pragma unroll
    for (int i = 0; i < kKeyLoads; ++i) {
      const int piece = tid + kThreads * i;
      const int key = piece / kChunks;
      const Octet o = f16x2::Split(key_next[i][0], key_next[i][1]);
      least.Add(f16x2::Largest(f16x2::Largest(0.0F, key_next[i][0]), key_next[i][1]));
      const int at = key * kKeyRow + piece % kChunks;
      key_planes[0][at] = o.h;
      key_planes[1][at] = o.l;
    }
    if (kValueThreads == kThreads || tid < kValueThreads) {
      const float4(&v)[4] = value_next;
      const float rows[4][4] = {{v[0].x, v[1].x, v[2].x, v[3].x},
                                {v[0].y, v[1].y, v[2].y, v[3].y},
                                {v[0].z, v[1].z, v[2].z, v[3].z},
                                {v[0].w, v[1].w, v[2].w, v[3].w}};
      // S^T leaves keys 16 c + 8 j + 4 half + 0..3 in one lane's registers:
      // the row holds, per 16 keys, half 0's two quads and then half 1's.
      const bool whole = key0 + 4 * value_quad + 4 <= key_end;
      const int slot = (value_quad / 4) * 32 + (value_quad % 2) * 16 + ((value_quad / 2) % 2) * 8;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f16x2::Pair p0 = f16x2::Split(rows[e][0], rows[e][1]);
        const f16x2::Pair p1 = f16x2::Split(rows[e][2], rows[e][3]);
        least.Add(f16x2::Largest(0.0F, v[e]));
        least.Add(whole ? f16x2::Largest(0.0F, make_float4(rows[e][0], rows[e][1], rows[e][2],
                                                           rows[e][3]))
                        : 0.0F);
        const int at = (4 * dim_quad + e) * kValueRow + slot;
        *reinterpret_cast<uint2*>(&value_planes[0][at]) = uint2{p0.h, p1.h};
        *reinterpret_cast<uint2*>(&value_planes[1][at]) = uint2{p0.l, p1.l};
      }
    }
  };

  if (tid == 0)
    restart = 0;
  load(key_begin);
  Octet qs[kSteps];
  {
    const float* source = a.q + static_cast<std::size_t>(place(query)) * D + 8 * half;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      float4 x = reinterpret_cast<const float4*>(source + 16 * s)[0];
      float4 y = reinterpret_cast<const float4*>(source + 16 * s)[1];
      x = make_float4(x.x * a.scale, x.y * a.scale, x.z * a.scale, x.w * a.scale);
      y = make_float4(y.x * a.scale, y.y * a.scale, y.z * a.scale, y.w * a.scale);
      qs[s] = f16x2::Split(x, y);
      least.Add(f16x2::Largest(f16x2::Largest(0.0F, x), y));
    }
  }

  F32x16 out[kTiles];
#pragma unroll
  for (int i = 0; i < kTiles; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v)
      out[i][v] = 0.0F;
  float maximum = -INFINITY;
  float sum = 0.0F;  // of this lane's keys

  for (int key0 = key_begin; key0 < key_end; key0 += kKeys) {
    __syncthreads();  // the step before has been read
    store(key0);
    __syncthreads();
    // Steps past the run's end load zeros.
    load(key0 + kKeys);
    if (key0 >= wave_keys)
      continue;

    F32x16 score;  // hh
    F32x16 cross;  // hl + lh, 2048 times their value
#pragma unroll
    for (int v = 0; v < 16; ++v)
      score[v] = cross[v] = 0.0F;
    const auto key_octet = [&](int s) {
      const int at = column * kKeyRow + 2 * s + half;
      return Octet{key_planes[0][at], key_planes[1][at]};
    };
    Octet ahead = key_octet(0);
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const Octet o = ahead;
      if (s + 1 < kSteps)
        ahead = key_octet(s + 1);
      __builtin_amdgcn_sched_barrier(0);  // read before the products it waits for
      cross = f16x2::Mfma32(o.l, qs[s].h, cross);
      score = f16x2::Mfma32(o.h, qs[s].h, score);
      cross = f16x2::Mfma32(o.h, qs[s].l, cross);
    }
    float p[16];
#pragma unroll
    for (int v = 0; v < 16; ++v)
      p[v] = __builtin_fmaf(cross[v], f16x2::kCross, score[v]);
    const bool masked = key0 + kKeys > whole_keys;
    if (masked) {
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (key0 + 8 * (v / 4) + 4 * half + v % 4 >= my_keys)
          p[v] = -INFINITY;
    }
    float top = p[0];
#pragma unroll
    for (int v = 1; v < 16; ++v)
      top = fmaxf(top, p[v]);
    top = fmaxf(maximum, MaxXor32(top));
    if (__any(top > maximum)) {
      // (-inf - top would make 2^(x log2 e)'s correction a NaN.)
      const float decay = maximum == -INFINITY ? 0.0F : ExpNegative(maximum - top);
      sum *= decay;
#pragma unroll
      for (int i = 0; i < kTiles; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          out[i][v] *= decay;
      maximum = top;
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const bool drop = masked && p[v] == -INFINITY;
      const float e = ExpNegative(drop ? 0.0F : p[v] - maximum);
      p[v] = drop ? 0.0F : e;
      sum += p[v];
    }
    Octet weights[2];
#pragma unroll
    for (int c = 0; c < 2; ++c)
      weights[c] = f16x2::Split(make_float4(p[8 * c], p[8 * c + 1], p[8 * c + 2], p[8 * c + 3]),
                                make_float4(p[8 * c + 4], p[8 * c + 5], p[8 * c + 6],
                                            p[8 * c + 7]));
#pragma unroll
    for (int i = 0; i < kTiles; ++i) {
      F32x16 apart;  // the cross terms
#pragma unroll
      for (int v = 0; v < 16; ++v)
        apart[v] = 0.0F;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int at = (32 * i + column) * kValueRow + 32 * c + 16 * half;
        const Octet o{*reinterpret_cast<const uint4*>(&value_planes[0][at]),
                      *reinterpret_cast<const uint4*>(&value_planes[1][at])};
        apart = f16x2::Mfma32(o.l, weights[c].h, apart);
        out[i] = f16x2::Mfma32(o.h, weights[c].h, out[i]);
        apart = f16x2::Mfma32(o.h, weights[c].l, apart);
      }
#pragma unroll
      for (int v = 0; v < 16; ++v)
        out[i][v] = __builtin_fmaf(apart[v], f16x2::kCross, out[i][v]);
    }
  }

  // 0, or NaN where a sum is NaN or infinite.
  float check[4] = {0.0F * sum, 0.0F, 0.0F, 0.0F};
#pragma unroll
  for (int i = 0; i < kTiles; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v)
      check[v % 4] = __builtin_fmaf(out[i][v], 0.0F, check[v % 4]);
  if (least.Below(kLeast) || check[0] + check[1] + (check[2] + check[3]) != 0.0F)
    restart = 1;
  __syncthreads();
  // Located again rather than held in registers through the steps (a spilled
  // one's reload waits for the loads in flight).
  int last_query = query;
  asm volatile("" : "+v"(last_query));
  const std::size_t at = static_cast<std::size_t>(place(last_query));
  if (restart != 0) {
    // Key by key in float32: each half of the wave takes half the dimensions
    // of a score, and its own of the values. Keys a query does not count are
    // left out, whatever they hold.
    maximum = -INFINITY;
    sum = 0.0F;
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        out[i][v] = 0.0F;
#pragma unroll 1
    for (int key = key_begin; key < key_end; ++key) {
      const float4* const k4 = reinterpret_cast<const float4*>(
          a.k + cache + static_cast<std::size_t>(key) * D + half * (D / 2));
      const float4* const q4 = reinterpret_cast<const float4*>(a.q + at * D + half * (D / 2));
      float dot = 0.0F;
#pragma unroll 1
      for (int i = 0; i < D / 8; ++i) {
        const float4 x = q4[i];
        const float4 y = k4[i];
        dot += x.x * a.scale * y.x + x.y * a.scale * y.y + x.z * a.scale * y.z +
               x.w * a.scale * y.w;
      }
      dot = AddXor32(dot);
      if (key >= my_keys)
        continue;
      const float top = fmaxf(maximum, dot);
      const float decay = maximum == -INFINITY ? 0.0F : expf(maximum - top);
      const float e = dot == -INFINITY ? 0.0F : expf(dot - top);
      maximum = top;
      sum = sum * decay + (half == 0 ? e : 0.0F);
      const float* const value = a.v + cache + static_cast<std::size_t>(key) * D + 4 * half;
#pragma unroll
      for (int i = 0; i < kTiles; ++i) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const float4 x = *reinterpret_cast<const float4*>(value + 32 * i + 8 * b);
          out[i][4 * b] = out[i][4 * b] * decay + e * x.x;
          out[i][4 * b + 1] = out[i][4 * b + 1] * decay + e * x.y;
          out[i][4 * b + 2] = out[i][4 * b + 2] * decay + e * x.z;
          out[i][4 * b + 3] = out[i][4 * b + 3] * decay + e * x.w;
        }
        __builtin_amdgcn_sched_barrier(0);  // one tile's values in registers
      }
    }
  }

  sum = AddXor32(sum);
  if (key_begin >= my_keys)
    return;  // past the last query, or before this chunk: nothing to leave
  // Element v of tile i: dimension 32 i + 8 (v / 4) + 4 half + v % 4.
  if (a.splits == 1) {
    const float inverse = 1.0F / sum;
    Bf16* target = a.out + at * D + 4 * half;
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        *reinterpret_cast<uint2*>(target + 32 * i + 8 * b) =
            uint2{q8::PackBf16x2(out[i][4 * b] * inverse, out[i][4 * b + 1] * inverse),
                  q8::PackBf16x2(out[i][4 * b + 2] * inverse, out[i][4 * b + 3] * inverse)};
    return;
  }
  float* target = a.values + (at * a.splits + split) * D + 4 * half;
#pragma unroll
  for (int i = 0; i < kTiles; ++i)
#pragma unroll
    for (int b = 0; b < 4; ++b)
      *reinterpret_cast<float4*>(target + 32 * i + 8 * b) =
          make_float4(out[i][4 * b], out[i][4 * b + 1], out[i][4 * b + 2], out[i][4 * b + 3]);
  if (half == 0) {
    float* stats = a.stats + (at * a.splits + split) * 2;
    stats[0] = maximum;
    stats[1] = sum;
  }
}

/// The chunks of a (row, head) met in chunk order: M = max m_c, L = sum
/// l_c exp(m_c - M), out = bf16(sum o_c exp(m_c - M) / L) over the row's
/// chunks. D / 4 lanes per (row, head), four dimensions each; lane c holds
/// chunk c's statistics (chunks D / 4 apart in turn), and the first chunks'
/// values are loaded beside them, so that they share a memory round trip (a
/// lane reading them chunk by chunk took 10.2 us for 300 rows of 16 heads
/// and 12 chunks, this 6.8).
template<int D>
__global__ __launch_bounds__(kThreads) void MergeChunksKernel(TileArgs a, int items) {
  constexpr int kLanes = D / 4;
  constexpr int kBatch = 8;
  const int item = static_cast<int>(blockIdx.x) * (kThreads / kLanes) +
                   static_cast<int>(threadIdx.x) / kLanes;
  if (item >= items)  // whole groups of lanes
    return;
  const int lane = static_cast<int>(threadIdx.x) % kLanes;
  const int local = (item / a.heads) % a.rows_per_sequence;
  const int keys = a.past + (a.causal != 0 ? local + 1 : a.rows_per_sequence);
  const int chunks = (keys + a.chunk - 1) / a.chunk;
  const std::size_t first = static_cast<std::size_t>(item) * a.splits;
  const float2* stats = reinterpret_cast<const float2*>(a.stats) + first;
  const float4* values = reinterpret_cast<const float4*>(a.values + first * D) + lane;
  float4 v[kBatch];
  const auto load = [&](int c0) {
#pragma unroll
    for (int b = 0; b < kBatch; ++b)
      v[b] = values[static_cast<std::size_t>(min(c0 + b, chunks - 1)) * kLanes];
  };
  load(0);
  const float2 mine = stats[min(lane, chunks - 1)];
  float top = mine.x;
  for (int c = lane + kLanes; c < chunks; c += kLanes)
    top = fmaxf(top, stats[c].x);
#pragma unroll
  for (int offset = kLanes / 2; offset > 0; offset /= 2)
    top = fmaxf(top, __shfl_xor(top, offset, kLanes));
  float4 out = make_float4(0.0F, 0.0F, 0.0F, 0.0F);
  float sum = 0.0F;
  for (int base = 0; base < chunks; base += kLanes) {
    const float2 s = base == 0 ? mine : stats[min(base + lane, chunks - 1)];
    const float factor = base + lane < chunks ? expf(s.x - top) : 0.0F;
    if (base + lane < chunks)
      sum += s.y * factor;
    const int count = min(kLanes, chunks - base);
    for (int c0 = 0; c0 < count; c0 += kBatch) {
      if (base + c0 > 0)
        load(base + c0);
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        const float f = __shfl(factor, c0 + b, kLanes);
        if (c0 + b < count) {
          out.x += v[b].x * f;
          out.y += v[b].y * f;
          out.z += v[b].z * f;
          out.w += v[b].w * f;
        }
      }
    }
  }
#pragma unroll
  for (int offset = kLanes / 2; offset > 0; offset /= 2)
    sum += __shfl_xor(sum, offset, kLanes);
  const float inverse = 1.0F / sum;
  *reinterpret_cast<uint2*>(a.out + static_cast<std::size_t>(item) * D + 4 * lane) =
      uint2{q8::PackBf16x2(out.x * inverse, out.y * inverse),
            q8::PackBf16x2(out.z * inverse, out.w * inverse)};
}

template<int D>
void Launch(const TileArgs& args, std::size_t workgroups, std::size_t items, hipStream_t stream) {
  TileAttentionKernel<D><<<static_cast<unsigned>(workgroups), kThreads, 0, stream>>>(args);
  if (args.splits > 1) {
    constexpr std::size_t kItems = kThreads / (D / 4);
    MergeChunksKernel<D><<<static_cast<unsigned>((items + kItems - 1) / kItems), kThreads, 0,
                           stream>>>(args, static_cast<int>(items));
  }
}

bool Aligned16(const void* p) { return reinterpret_cast<std::uintptr_t>(p) % 16 == 0; }

}  // namespace

bool PlanTileAttention(const AttentionShape& s, const float* q, const float* k_cache,
                       const float* v_cache, const Bf16* out, const float* partials,
                       TileAttentionPlan* plan) {
  const std::size_t group = s.heads / s.kv_heads;
  // The kernel's indices are 32-bit; the caches are read in 16-byte pieces.
  if (s.rows_per_sequence * group < 32 || s.rows * s.heads >= (std::size_t{1} << 24) ||
      s.past + s.rows_per_sequence >= (std::size_t{1} << 21) || !Aligned16(q) ||
      !Aligned16(k_cache) || !Aligned16(v_cache) || !Aligned16(out) || !Aligned16(partials))
    return false;
  const std::size_t queries = s.rows_per_sequence * group;
  const std::size_t blocks = (queries + kQueries - 1) / kQueries;
  const std::size_t heads = s.rows / s.rows_per_sequence * s.kv_heads;
  const auto keys_of = [&](std::size_t block) {
    const std::size_t last = std::min((block + 1) * kQueries, queries) - 1;
    return s.past + (s.causal ? last / group + 1 : s.rows_per_sequence);
  };
  const auto runs_of = [&](std::size_t chunk) {
    std::size_t runs = 0;
    for (std::size_t b = 0; b < blocks; ++b)
      runs += (keys_of(b) + chunk - 1) / chunk;
    return runs * heads;
  };
  // The least chunk that cuts all query blocks' keys into at most
  // kTargetWorkgroups runs (or leaves them whole).
  std::size_t steps = 0;
  for (std::size_t b = 0; b < blocks; ++b)
    steps += (keys_of(b) + kKeys - 1) / kKeys;
  const std::size_t most = s.past + s.rows_per_sequence;
  std::size_t chunk = std::max<std::size_t>(
      kLeastChunk, (steps * heads + kTargetWorkgroups - 1) / kTargetWorkgroups * kKeys);
  while (chunk < most && runs_of(chunk) > kTargetWorkgroups)
    chunk += kKeys;
  plan->chunk = chunk;
  plan->splits = (most + chunk - 1) / chunk;
  plan->workgroups = plan->splits == 1 ? blocks * heads : runs_of(chunk);
  return true;
}

bool UseTileAttention(const AttentionShape& s, const TileAttentionPlan& plan, int splits,
                      int heads_per_workgroup) {
  // Both kernels' times in microseconds, fitted to MI355X over rows 4..3000, keys
  // 2..3260, groups 1..16 and head_dim 64 and 128 (2924 points, replayed from a
  // graph): here a workgroup's steps of 32 keys in its round of two workgroups
  // per compute unit, there the rounds of one per unit, the longer the more
  // heads each scores, and a merge each. The choice takes on average 0.5 % longer
  // than the faster kernel, one in eighty over 5 % longer than the split
  // kernel. 4 rows of 16 heads over 254 keys 7.6 us there, 16.4 here; 64 rows 5.7
  // and 11.2, 65 rows (a second chunk and round) 16.4 and 11.1; 16 rows over 716
  // keys 16.2 and 19.5; 64 over 314 22.8 and 19.6; 128 over 828 81.7 and 23.1; 40
  // patches of 5 rows 13.2 and 6.9.
  const bool wide = s.head_dim > 64;
  const std::size_t keys = std::min(plan.chunk, s.past + s.rows_per_sequence);
  const double steps = static_cast<double>((keys + kKeys - 1) / kKeys);
  const double here =
      4.2 + (plan.splits > 1 ? 4.4 : 0.0) +
      static_cast<double>((plan.workgroups + kTargetWorkgroups - 1) / kTargetWorkgroups) * steps *
          (wide ? 2.65 : 1.6);
  const std::size_t workgroups =
      s.rows * s.heads / heads_per_workgroup * static_cast<std::size_t>(splits);
  const double there = 2.8 + (splits > 1 ? 3.2 : 0.0) +
                       static_cast<double>((workgroups + 255) / 256) *
                           (wide ? 0.68 + 0.49 * heads_per_workgroup
                                 : 0.28 + 0.16 * heads_per_workgroup);
  return here < there;
}

void TileAttention(const AttentionShape& s, const TileAttentionPlan& plan, const float* q,
                   const float* k_cache, const float* v_cache, Bf16* out, float* partials,
                   hipStream_t stream) {
  const std::size_t group = s.heads / s.kv_heads;
  const std::size_t queries = s.rows_per_sequence * group;
  TileArgs args{};
  args.q = q;
  args.k = k_cache;
  args.v = v_cache;
  args.out = out;
  args.values = partials;
  args.stats = partials == nullptr ? nullptr : partials + s.rows * s.heads * plan.splits * s.head_dim;
  args.rows_per_sequence = static_cast<int>(s.rows_per_sequence);
  args.keys_per_sequence = static_cast<int>(s.keys_per_sequence);
  args.past = static_cast<int>(s.past);
  args.causal = s.causal ? 1 : 0;
  args.heads = static_cast<int>(s.heads);
  args.kv_heads = static_cast<int>(s.kv_heads);
  args.capacity = static_cast<int>(s.capacity);
  args.sequences = static_cast<int>(s.rows / s.rows_per_sequence);
  args.blocks = static_cast<int>((queries + kQueries - 1) / kQueries);
  args.chunk = static_cast<int>(plan.chunk);
  args.splits = static_cast<int>(plan.splits);
  args.scale = 1.0F / std::sqrt(static_cast<float>(s.head_dim));
  const std::size_t items = s.rows * s.heads;
  if (s.head_dim == 64)
    Launch<64>(args, plan.workgroups, items, stream);
  else
    Launch<128>(args, plan.workgroups, items, stream);
}

}  // namespace vx
