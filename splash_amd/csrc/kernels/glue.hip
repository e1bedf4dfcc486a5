// Glue kernels of the verify path: RMS norm (with the projection's activation table fused in),
// RoPE tables per packed row, token embedding from native K-quant rows (the reference's
// kernels/shared/normalization.metal, rope.metal, embedding.metal).
#include "abi/Glue.h"
#include "abi/DraftAttention.h"
#include "abi/Gguf.h"
#include "backend/KernelRegistry.hpp"
#include "kernels/device_common.hpp"

#include <type_traits>

namespace splash::kernels {

// Rows of up to kStagedWidth columns are staged in LDS with every global load in flight at once
// (a row's columns are read twice, in an order no vector load gives directly).
constexpr uint32_t kStagedWidth = NORM_STAGED_WIDTH;

// `v` has arrived: nothing that uses it moves above this, and its load does not move below. A load that is sunk to its use
// under a condition is waited for alone, one round trip each.
__device__ __forceinline__ void arrived(uint4 &v) { asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w)); }
__device__ __forceinline__ void arrived(uint32_t &v) { asm volatile("" : "+v"(v)); }

// `width` bf16 values (a multiple of 8, 16-byte aligned) on their way to LDS: every load of it goes out before any is stored,
// and those of several rows before the first row's stores. No barrier. (A norm of 8 rows of 5120: 8.7 us where each load was
// waited for, 7.9 with the loads unconditional but sunk to their stores, 6.6 so.)
struct StagedRow {
  static constexpr uint32_t kHeld = kStagedWidth / 8u / 256u;
  uint4 held[kHeld];
  __device__ __forceinline__ void load(const uint16_t *__restrict__ source, uint32_t width) {
#pragma unroll
    for (uint32_t i = 0; i < kHeld; ++i)   // (the last vector again past the row's end)
      held[i] = reinterpret_cast<const uint4 *>(source)[min(threadIdx.x + 256u * i, width / 8u - 1u)];
  }
  __device__ __forceinline__ void store(uint32_t width, uint16_t *lds) {
#pragma unroll
    for (uint32_t i = 0; i < kHeld; ++i) arrived(held[i]);
#pragma unroll
    for (uint32_t i = 0; i < kHeld; ++i) {
      const uint32_t v = threadIdx.x + 256u * i;
      if (v < width / 8u) reinterpret_cast<uint4 *>(lds)[v] = held[i];
    }
  }
};

__global__ __launch_bounds__(256) void norm_rms(const uint16_t *__restrict__ input, const uint16_t *__restrict__ weight,
                                                uint16_t *__restrict__ output, NormParams p) {
  __shared__ float scratch[4];
  __shared__ __align__(16) uint16_t rowX[kStagedWidth], rowW[kStagedWidth];
  const uint32_t row = blockIdx.x;
  const uint16_t *x = input + size_t(row) * p.width, *w = weight;
  if (p.width <= kStagedWidth && p.width % 8u == 0) {
    StagedRow stagedX, stagedW;
    stagedX.load(x, p.width);
    stagedW.load(w, p.width);
    stagedX.store(p.width, rowX);
    stagedW.store(p.width, rowW);
    __syncthreads();
    x = rowX;
    w = rowW;
  }
  const float inverse = rms_inverse(x, p.width, scratch);
  for (uint32_t c = threadIdx.x; c < p.width; c += 256)
    output[size_t(row) * p.width + c] = uint16_t(float_to_bf16_bits((bf16_bits_to_float(x[c]) * inverse) * bf16_bits_to_float(w[c])));
}
SP_REGISTER_KERNEL("norm_rms", &norm_rms);

// A row's part of an activation table, and the normalized row it describes, of rows wider than kStagedWidth: 256 threads,
// each the runs of four inputs q = t, t + 256, ... (4 kq .. 4 kq + 3 of a group's half, one 8-byte piece of a table entry),
// kRuns of them in flight together. A row past the live ones is zeros. The width is a multiple of 256, so a wavefront's runs
// are all inside the row or all past it.
__device__ __forceinline__ void write_table_row(const uint16_t *x, const uint16_t *w, float inverse, bool live, uint32_t row,
                                                uint16_t *__restrict__ output, uint8_t *__restrict__ table, uint32_t width, uint32_t allTiles) {
  constexpr uint32_t kRuns = 5;
  const uint32_t r = row % 16u, G = width / 32u, runs = width / 4u;
  // Row tile row / 16 is tile `tile` of its piece's table, which holds `tiles` row tiles.
  const uint32_t piece = row / 16u / GGUF_PIECE_TILES, tile = row / 16u % GGUF_PIECE_TILES;
  const uint32_t tiles = min(uint32_t(GGUF_PIECE_TILES), allTiles - piece * GGUF_PIECE_TILES);
  table += piece * gguf_table_bytes(width, GGUF_PIECE_TILES);
  uint2 *values = reinterpret_cast<uint2 *>(table);
  float *sums32 = reinterpret_cast<float *>(table + gguf_table_sums32_offset(width, tiles));
  float *sums16 = reinterpret_cast<float *>(table + gguf_table_sums16_offset(width, tiles));
  for (uint32_t first = 0; first < runs; first += 256u * kRuns) {
    uint32_t bits[kRuns][4];
    float sum[kRuns];
#pragma unroll
    for (uint32_t j = 0; j < kRuns; ++j) {
      const uint32_t q = min(first + 256u * j + threadIdx.x, runs - 1u);
      uint2 xs = make_uint2(0u, 0u), ws = xs;
      if (live) {
        xs = *reinterpret_cast<const uint2 *>(x + 4u * q);
        ws = *reinterpret_cast<const uint2 *>(w + 4u * q);
      }
      const uint32_t xb[4] = {xs.x & 0xFFFFu, xs.x >> 16, xs.y & 0xFFFFu, xs.y >> 16};
      const uint32_t wb[4] = {ws.x & 0xFFFFu, ws.x >> 16, ws.y & 0xFFFFu, ws.y >> 16};
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bits[j][i] = live ? float_to_bf16_bits((bf16_bits_to_float(xb[i]) * inverse) * bf16_bits_to_float(wb[i])) : 0u;
        v[i] = bf16_bits_to_float(bits[j][i]);
      }
      sum[j] = (v[0] + v[1]) + (v[2] + v[3]);
    }
#pragma unroll
    for (uint32_t j = 0; j < kRuns; ++j) {
      const uint32_t q = first + 256u * j + threadIdx.x;
      // run q: group g = q / 8, half = (q / 4) % 2, kq = q % 4; the four runs of a half sit in four consecutive lanes
      const float s1 = lane_down<1>(sum[j]), s2 = lane_down<2>(sum[j]), s3 = lane_down<3>(sum[j]);
      const float s = ((sum[j] + s1) + s2) + s3;   // of 16 inputs, in input order
      const float other = lane_down<4>(s);
      if (q >= runs) continue;
      if (live)
        *reinterpret_cast<uint2 *>(output + size_t(row) * width + 4u * q) =
            make_uint2(bits[j][0] | (bits[j][1] << 16), bits[j][2] | (bits[j][3] << 16));
      const uint32_t g = q / 8u, half = (q / 4u) % 2u, kq = q % 4u;
      // operand elements 4 half + {0,1,2,3} are inputs 4 kq + {0,2,1,3} of the half
      values[((size_t(tile) * G + g) * 64u + kq * 16u + r) * 2u + half] =
          make_uint2(bits[j][0] | (bits[j][2] << 16), bits[j][1] | (bits[j][3] << 16));
      if (kq == 0) {
        sums16[(size_t(tile) * 2u * G + 2u * g + half) * 16u + r] = s;
        if (half == 0) sums32[(size_t(tile) * G + g) * 16u + r] = s + other;
      }
    }
  }
}

// Eight inputs 8 v .. 8 v + 7 of a row, a thread of its own for each v: their two pieces of the row's activation table and
// their parts of its sums, the values and the order of additions of write_table_row. Lanes 4 l .. 4 l + 3 hold consecutive v
// of one group of 32 inputs.
__device__ __forceinline__ void write_table_vector(uint4 bits, uint32_t row, uint32_t v, uint8_t *__restrict__ table, uint32_t width, uint32_t allTiles) {
  const uint32_t r = row % 16u, G = width / 32u;
  const uint32_t piece = row / 16u / GGUF_PIECE_TILES, tile = row / 16u % GGUF_PIECE_TILES;
  const uint32_t tiles = min(uint32_t(GGUF_PIECE_TILES), allTiles - piece * GGUF_PIECE_TILES);
  table += piece * gguf_table_bytes(width, GGUF_PIECE_TILES);
  uint2 *values = reinterpret_cast<uint2 *>(table);
  const uint32_t g = v / 4u, half = (v / 2u) % 2u, kq = 2u * (v % 2u);
  auto four = [](uint32_t low, uint32_t high) {
    return (bf16_bits_to_float(low & 0xFFFFu) + bf16_bits_to_float(low >> 16)) + (bf16_bits_to_float(high & 0xFFFFu) + bf16_bits_to_float(high >> 16));
  };
  const float a = four(bits.x, bits.y), b = four(bits.z, bits.w), a1 = lane_down<1>(a), b1 = lane_down<1>(b);
  const float s = ((a + b) + a1) + b1;   // of 16 inputs, in input order
  const float other = lane_down<2>(s);
  // operand elements 4 half + {0,1,2,3} are inputs 4 kq + {0,2,1,3} of the half
  auto operand = [](uint32_t low, uint32_t high) { return make_uint2((low & 0xFFFFu) | (high << 16), (low >> 16) | (high & 0xFFFF0000u)); };
  uint2 *at = values + ((size_t(tile) * G + g) * 64u + kq * 16u + r) * 2u + half;
  at[0] = operand(bits.x, bits.y);
  at[32] = operand(bits.z, bits.w);
  if (kq == 0) {
    float *sums32 = reinterpret_cast<float *>(table + gguf_table_sums32_offset(width, tiles));
    float *sums16 = reinterpret_cast<float *>(table + gguf_table_sums16_offset(width, tiles));
    sums16[(size_t(tile) * 2u * G + 2u * g + half) * 16u + r] = s;
    if (half == 0) sums32[(size_t(tile) * G + g) * 16u + r] = s + other;
  }
}

// Eight values of a normalized row.
__device__ __forceinline__ uint4 norm_vector(uint4 x, uint4 w, float inverse) {
  auto two = [&](uint32_t xs, uint32_t ws) {
    const uint32_t low = float_to_bf16_bits((bf16_bits_to_float(xs & 0xFFFFu) * inverse) * bf16_bits_to_float(ws & 0xFFFFu));
    return low | (float_to_bf16_bits((bf16_bits_to_float(xs >> 16) * inverse) * bf16_bits_to_float(ws >> 16)) << 16);
  };
  return make_uint4(two(x.x, w.x), two(x.y, w.y), two(x.z, w.z), two(x.w, w.w));
}
// Eight values of a normalized row and their part of the table; zeros in the table for a row past the live ones. (Eight bytes
// a store: all that the rows' buffers promise.)
__device__ __forceinline__ void write_norm_vector(uint4 x, uint4 w, float inverse, bool live, uint32_t row, uint32_t v, uint16_t *__restrict__ output,
                                                  uint8_t *__restrict__ table, uint32_t width, uint32_t tiles) {
  uint4 bits = make_uint4(0u, 0u, 0u, 0u);
  if (live) {
    bits = norm_vector(x, w, inverse);
    uint2 *to = reinterpret_cast<uint2 *>(output + size_t(row) * width + 8u * v);
    to[0] = make_uint2(bits.x, bits.y);
    to[1] = make_uint2(bits.z, bits.w);
  }
  write_table_vector(bits, row, v, table, width, tiles);
}

// A row's normalized vectors by a workgroup: a thread's first from its registers (its values and weights), those past it, where
// the workgroup has fewer threads than the row has vectors, from LDS and memory.
__device__ __forceinline__ void write_norm_vectors(uint4 mine, uint4 norm, const uint16_t *row_x, const uint16_t *__restrict__ weight, float inverse,
                                                   bool live, uint32_t row, uint16_t *__restrict__ output, uint8_t *__restrict__ table,
                                                   uint32_t width, uint32_t tiles) {
  const uint32_t vectors = width / 8u, first = threadIdx.x;
  if (first < vectors) write_norm_vector(mine, norm, inverse, live, row, first, output, table, width, tiles);
  for (uint32_t v = first + blockDim.x; v < vectors; v += blockDim.x) {
    if (live) norm = reinterpret_cast<const uint4 *>(weight)[v];
    write_norm_vector(reinterpret_cast<const uint4 *>(row_x)[v], norm, inverse, live, row, v, output, table, width, tiles);
  }
}

// The same, and the activation table of the normalized rows: grid (tiles * 16) so that the rows past the live ones are
// written as zeros, norm_row_threads(width) threads (any whole wavefronts from 256 threads on are right). A handful of workgroups that only wait, so what counts is the chain one
// thread runs: a row of up to kStagedWidth columns has a thread a vector of eight, which holds it and its weights in
// registers from the load to the stores, and LDS serves the sum alone. (8 rows of 5120: 7.4 us by 256 threads, 4.3 so; 128 of
// 2048: 6.0 and 5.6.)
__global__ __launch_bounds__(1024) void norm_rms_table16(const uint16_t *__restrict__ input, const uint16_t *__restrict__ weight,
                                                         uint16_t *__restrict__ output, uint8_t *__restrict__ table, NormParams p) {
  __shared__ float scratch[4];
  __shared__ __align__(16) uint16_t rowX[kStagedWidth];
  const uint32_t row = blockIdx.x;
  const bool live = row < p.rows;
  const uint16_t *x = input + size_t(live ? row : 0) * p.width;
  if (p.width <= kStagedWidth) {  // the width is a multiple of 256
    const uint32_t vectors = p.width / 8u, first = threadIdx.x;
    uint4 mine = make_uint4(0u, 0u, 0u, 0u), norm = mine;
    if (live) {
      if (first < vectors) {
        mine = reinterpret_cast<const uint4 *>(x)[first];
        norm = reinterpret_cast<const uint4 *>(weight)[first];
        reinterpret_cast<uint4 *>(rowX)[first] = mine;
      }
      for (uint32_t v = first + blockDim.x; v < vectors; v += blockDim.x) reinterpret_cast<uint4 *>(rowX)[v] = reinterpret_cast<const uint4 *>(x)[v];
    }
    __syncthreads();
    const float inverse = live ? rms_inverse(rowX, p.width, scratch) : 0.f;
    write_norm_vectors(mine, norm, rowX, weight, inverse, live, row, output, table, p.width, p.tiles);
  } else {
    const float inverse = live ? rms_inverse(x, p.width, scratch) : 0.f;
    write_table_row(x, weight, inverse, live, row, output, table, p.width, p.tiles);
  }
}
SP_REGISTER_KERNEL("norm_rms_table16", &norm_rms_table16);

// draft_conv (draft_attention.hip) and the pass that reads its rows, a thread a vector of eight channels: a Prepare stage's
// rows and their activation table, grid (tiles * 16, the row's vectors by 64), 64 threads, since nothing there needs the
// row's other channels; a Residual stage's rows, their RMS norm (of `norm_weight`, into `normalized`) and its table, a
// workgroup of norm_row_threads(width) a row. (A launch of fewer threads, of the one any, of the other whole 256, takes its
// vectors in turns.) Each convolution was a launch of its own before a launch of as few workgroups.
// 8 rows of 5120, inside a draft model's pass: 3.1 us (a workgroup of 256 a row, 5.3) and 4.7 (8.3).
// Values and their order are the two kernels'. The rows' 16-byte accesses are the host's rule
// (DraftAttention::addConvolutionTable).
template <bool Residual>
__global__ __launch_bounds__(Residual ? 1024 : 256) void draft_conv_table(
    const uint16_t *__restrict__ input, const uint16_t *__restrict__ dynamic, const uint16_t *__restrict__ base,
    const uint16_t *__restrict__ residual, const uint16_t *__restrict__ norm_weight, uint16_t *__restrict__ output,
    uint16_t *__restrict__ normalized, uint8_t *__restrict__ table, DraftConvTableParams p) {
  static_assert(DRAFT_CONVOLUTION_TABLE_WIDTH <= kStagedWidth && DRAFT_CONVOLUTION_GROUP % 8u == 0, "eight channels share their dynamic weights");
  __shared__ float scratch[4];
  __shared__ __align__(16) uint16_t rowX[Residual ? kStagedWidth : 8];
  const uint32_t row = blockIdx.x, width = p.hidden, vectors = width / 8u, groups = width / DRAFT_CONVOLUTION_GROUP;
  const uint32_t start = Residual ? threadIdx.x : blockIdx.y * 64u + threadIdx.x;
  const bool live = row < p.rows;
  uint4 norm = make_uint4(0u, 0u, 0u, 0u);
  auto convolve = [&](uint32_t v) __attribute__((always_inline)) {
    const bool follows = row % DRAFT_ATTENTION_QUERY_ROWS > 0;   // a lane's first row has none before it
    const size_t before = row - (follows ? 1u : 0u);
    const uint16_t *mine = dynamic + size_t(row) * draft_dynamic_width(width) + (Residual ? DRAFT_CONVOLUTION_TAPS : 0u) * groups;
    const uint16_t *taps = base + (Residual ? DRAFT_CONVOLUTION_TAPS : 0u) * size_t(width);
    auto vector = [&](const uint16_t *from) { return reinterpret_cast<const uint4 *>(from)[v]; };
    uint4 now = vector(input + size_t(row) * width), last = vector(input + before * width), tap0 = vector(taps), tap1 = vector(taps + width);
    uint4 added = make_uint4(0u, 0u, 0u, 0u);
    if constexpr (Residual) added = vector(residual + size_t(row) * width);
    uint32_t dynamic0 = mine[v / (DRAFT_CONVOLUTION_GROUP / 8u)], dynamic1 = mine[groups + v / (DRAFT_CONVOLUTION_GROUP / 8u)];
    if constexpr (Residual)
      if (v == start) norm = vector(norm_weight);
    arrived(now);
    arrived(last);
    arrived(tap0);
    arrived(tap1);
    if constexpr (Residual) arrived(added);
    arrived(dynamic0);
    arrived(dynamic1);
    const float d0 = bf16_bits_to_float(dynamic0), d1 = bf16_bits_to_float(dynamic1);
    auto channel = [&](uint32_t x, uint32_t y, uint32_t t0, uint32_t t1, uint32_t a) {
      float value = bf16_bits_to_float(x) * (bf16_bits_to_float(t0) + d0);
      if (follows) value += bf16_bits_to_float(y) * (bf16_bits_to_float(t1) + d1);
      if constexpr (Residual) value += bf16_bits_to_float(a);
      return float_to_bf16_bits(value);
    };
    auto pair = [&](uint32_t x, uint32_t y, uint32_t t0, uint32_t t1, uint32_t a) {
      return channel(x & 0xFFFFu, y & 0xFFFFu, t0 & 0xFFFFu, t1 & 0xFFFFu, a & 0xFFFFu) | (channel(x >> 16, y >> 16, t0 >> 16, t1 >> 16, a >> 16) << 16);
    };
    const uint4 packed = make_uint4(pair(now.x, last.x, tap0.x, tap1.x, added.x), pair(now.y, last.y, tap0.y, tap1.y, added.y),
                                    pair(now.z, last.z, tap0.z, tap1.z, added.z), pair(now.w, last.w, tap0.w, tap1.w, added.w));
    reinterpret_cast<uint4 *>(output + size_t(row) * width)[v] = packed;
    if constexpr (Residual) reinterpret_cast<uint4 *>(rowX)[v] = packed;
    return packed;
  };
  const uint4 none = make_uint4(0u, 0u, 0u, 0u);
  if constexpr (Residual) {
    const uint4 mine = live && start < vectors ? convolve(start) : none;
    if (live)
      for (uint32_t v = start + blockDim.x; v < vectors; v += blockDim.x) convolve(v);
    __syncthreads();
    const float inverse = live ? rms_inverse(rowX, width, scratch) : 0.f;
    write_norm_vectors(mine, norm, rowX, norm_weight, inverse, live, row, normalized, table, width, p.tiles);
  } else {
    // (64 vectors a workgroup and turn, whatever its threads: more of them than 64 do the next turn's again)
    if (start < vectors) write_table_vector(live ? convolve(start) : none, row, start, table, width, p.tiles);
    for (uint32_t v = start + 64u * gridDim.y; v < vectors; v += 64u * gridDim.y)
      write_table_vector(live ? convolve(v) : none, row, v, table, width, p.tiles);
  }
}
SP_REGISTER_KERNEL("draft_conv_table", &draft_conv_table<false>);
SP_REGISTER_KERNEL("draft_conv_norm_table", &draft_conv_table<true>);

// copy_rows_bf16: grid (ceil(rows * width / 256)), 256 threads.
__global__ __launch_bounds__(256) void copy_rows_bf16(const uint16_t *__restrict__ source, uint16_t *__restrict__ destination, RowCopyParams p) {
  const uint64_t index = uint64_t(blockIdx.x) * 256u + threadIdx.x;
  if (index >= uint64_t(p.rows) * p.width) return;
  const uint32_t row = uint32_t(index / p.width), column = uint32_t(index % p.width);
  destination[(size_t(p.to_row) + row) * p.to_stride + p.to_column + column] =
      source[(size_t(p.from_row) + row) * p.from_stride + p.from_column + column];
}
SP_REGISTER_KERNEL("copy_rows_bf16", &copy_rows_bf16);

__global__ __launch_bounds__(256) void swiglu_rows(const uint16_t *__restrict__ gate, const uint16_t *__restrict__ up,
                                                   uint16_t *__restrict__ output, SwiGluRowsParams p) {
  const uint64_t first = (uint64_t(blockIdx.x) * 256u + threadIdx.x) * 8u;
  if (first >= p.count) return;
  if (first + 8u <= p.count) {
    const uint4 g = *reinterpret_cast<const uint4 *>(gate + first), u = *reinterpret_cast<const uint4 *>(up + first);
    const uint32_t gw[4] = {g.x, g.y, g.z, g.w}, uw[4] = {u.x, u.y, u.z, u.w};
    uint32_t out[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t low = float_to_bf16_bits(bf16_bits_to_float(uw[i] & 0xFFFFu) * silu(bf16_bits_to_float(gw[i] & 0xFFFFu)));
      const uint32_t high = float_to_bf16_bits(bf16_bits_to_float(uw[i] >> 16) * silu(bf16_bits_to_float(gw[i] >> 16)));
      out[i] = low | (high << 16);
    }
    *reinterpret_cast<uint4 *>(output + first) = make_uint4(out[0], out[1], out[2], out[3]);
  } else {
    for (uint64_t i = first; i < p.count; ++i)
      output[i] = uint16_t(float_to_bf16_bits(bf16_bits_to_float(up[i]) * silu(bf16_bits_to_float(gate[i]))));
  }
}
SP_REGISTER_KERNEL("swiglu_rows", &swiglu_rows);

__device__ __forceinline__ void rope_entry_at(uint32_t position, uint32_t row, uint32_t pair, const float *__restrict__ inverse_frequency,
                                              float *__restrict__ cosines, float *__restrict__ sines, uint32_t pairs) {
  const float angle = float(position) * inverse_frequency[pair];
  cosines[size_t(row) * pairs + pair] = cosf(angle);
  sines[size_t(row) * pairs + pair] = sinf(angle);
}
__device__ __forceinline__ void rope_entry(uint32_t row, uint32_t pair, const float *__restrict__ inverse_frequency,
                                           const uint32_t *__restrict__ depth, float *__restrict__ cosines, float *__restrict__ sines,
                                           const RopeTreeParams &p) {
  uint32_t anchor = 0;
  for (uint32_t s = 0; s < p.sequences; ++s)
    if (row >= p.first_row[s] && row < p.first_row[s] + p.row_count[s]) anchor = p.anchor[s];
  rope_entry_at(anchor + depth[row], row, pair, inverse_frequency, cosines, sines, p.pairs);
}
__global__ void rope_build_tree_tables(const float *__restrict__ inverse_frequency, const uint32_t *__restrict__ depth,
                                       float *__restrict__ cosines, float *__restrict__ sines, RopeTreeParams p) {
  const uint32_t row = blockIdx.x, pair = threadIdx.x;
  if (row < p.rows && pair < p.pairs) rope_entry(row, pair, inverse_frequency, depth, cosines, sines, p);
}
SP_REGISTER_KERNEL("rope_build_tree_tables", &rope_build_tree_tables);

// A prompt chunk's tables in one dispatch, whose blocks need no list of sequences: eight blocks a dispatch, 4.3 us each of
// which most is the launch, were 68 us of a 2048-row chunk.
__global__ __launch_bounds__(256) void rope_build_chunk_tables(const float *__restrict__ inverse_frequency, const uint32_t *__restrict__ depth,
                                                              float *__restrict__ cosines, float *__restrict__ sines, RopeChunkParams p) {
  const uint64_t at = uint64_t(blockIdx.x) * 256u + threadIdx.x;
  const uint32_t row = uint32_t(at / p.pairs), pair = uint32_t(at % p.pairs);
  if (row >= p.rows) return;
  rope_entry_at(p.anchor + row / p.block_rows * p.block_rows + depth[row], row, pair, inverse_frequency, cosines, sines, p.pairs);
}
SP_REGISTER_KERNEL("rope_build_chunk_tables", &rope_build_chunk_tables);

// gguf_float_<weights>_<output>: the fp32 projection of weights kept as rows (abi/Glue.h; the reference's
// kernels/shared/gguf_float.metal): a workgroup owns 16 rows x 16 columns and walks K in steps of 64 inputs staged in
// LDS (the rows' bf16 values widened, the weights as stored or widened: every operand exact in fp32); thread (r, c)
// runs the four chains of its output. The weights' rows are padded by one word in LDS so that the sixteen columns a
// half-wave reads at one input fall in sixteen banks.
template <bool kBf16Weights, bool kBf16Output>
__global__ __launch_bounds__(256) void gguf_float(const uint16_t *__restrict__ input, const void *__restrict__ weights,
                                                   void *__restrict__ output, GgufFloatParams p) {
  constexpr uint32_t S = GGUF_FLOAT_STEP;
  __shared__ float xs[16][S], ws[16][S + 1];
  const uint32_t tid = threadIdx.x, c = tid & 15u, r = tid >> 4;
  const uint32_t column0 = blockIdx.x * 16u, row0 = blockIdx.y * 16u, K = p.input_size;
  float chain[4] = {0.f, 0.f, 0.f, 0.f};
  for (uint32_t k0 = 0; k0 < K; k0 += S) {
    // stage: thread t the four inputs 4 (t % 16) .. of row / column t / 16; zeros past the rows, the columns and K
    {
      const uint32_t line = tid >> 4, at = (tid & 15u) * 4u;
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t k = k0 + at + i;
        const bool inside = k < K;
        float x = 0.f, w = 0.f;
        if (inside && row0 + line < p.rows) x = bf16_bits_to_float(input[size_t(row0 + line) * K + k]);
        if (inside && column0 + line < p.output_size) {
          if constexpr (kBf16Weights) w = bf16_bits_to_float(static_cast<const uint16_t *>(weights)[size_t(column0 + line) * K + k]);
          else w = static_cast<const float *>(weights)[size_t(column0 + line) * K + k];
        }
        xs[line][at + i] = x;
        ws[line][at + i] = w;
      }
    }
    __syncthreads();
#pragma unroll 4
    for (uint32_t k = 0; k < S; k += 4) {
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) chain[j] = __builtin_fmaf(xs[r][k + j], ws[c][k + j], chain[j]);
    }
    __syncthreads();
  }
  const float sum = (chain[0] + chain[1]) + (chain[2] + chain[3]);
  if (row0 + r >= p.rows || column0 + c >= p.output_size) return;
  const size_t at = size_t(row0 + r) * p.out_stride + p.out_offset + column0 + c;
  if constexpr (kBf16Output) static_cast<uint16_t *>(output)[at] = uint16_t(float_to_bf16_bits(sum));
  else static_cast<float *>(output)[at] = sum;
}
SP_REGISTER_KERNEL("gguf_float_f32_f32", (&gguf_float<false, false>));
SP_REGISTER_KERNEL("gguf_float_f32_bf16", (&gguf_float<false, true>));
SP_REGISTER_KERNEL("gguf_float_bf16_f32", (&gguf_float<true, false>));
SP_REGISTER_KERNEL("gguf_float_bf16_bf16", (&gguf_float<true, true>));

// Input k of a native super-block of 256 (embedding.metal:10-18).
template <uint32_t FMT> struct EmbedBlock {
  static constexpr uint32_t kBytes = FMT == GGUF_FMT_Q4K ? GGUF_Q4K_NATIVE : FMT == GGUF_FMT_Q5K ? GGUF_Q5K_NATIVE : FMT == GGUF_FMT_Q6K ? GGUF_Q6K_NATIVE
                                   : FMT == GGUF_FMT_Q80 ? GGUF_Q80_NATIVE : FMT == GGUF_FMT_IQ4XS ? GGUF_IQ4XS_NATIVE : GGUF_IQ4NL_NATIVE;
  static __device__ __forceinline__ uint32_t bits(const uint8_t *__restrict__ blk, uint32_t k) {
    const uint32_t j = k / 32u, e = k % 32u;
    if constexpr (FMT == GGUF_FMT_Q4K || FMT == GGUF_FMT_Q5K) {
      constexpr bool kFifth = FMT == GGUF_FMT_Q5K;   // Q5_K: 32 bytes of fifth bits between the scales and the nibbles
      const float d = half_bits_to_float(blk[0] | (blk[1] << 8)), dmin = half_bits_to_float(blk[2] | (blk[3] << 8));
      const uint8_t *sc = blk + 4, *qh = blk + 16, *qs = blk + (kFifth ? 48 : 16);
      // groups 0..3: six bits of bytes j and j + 4; groups 4..7: the halves of byte j + 4 and two bits of bytes j - 4 and j
      // (by masks, so that no branch stands between a thread's loads)
      const bool low = j < 4u;
      const uint32_t keep = low ? 63u : 15u, top = low ? 0u : 48u, shift = low ? 0u : 4u, both = sc[j + 4u];
      const uint32_t s = (sc[j + shift] & keep) | ((sc[j & 3u] >> 2) & top), m = ((both >> shift) & keep) | ((sc[(j & 3u) + 4u] >> 2) & top);
      uint32_t code = (qs[32u * (j / 2u) + e] >> (4u * (j % 2u))) & 15u;
      if constexpr (kFifth) code |= ((qh[e] >> j) & 1u) << 4;
      return float_to_bf16_bits(__fmaf_rn(d * float(s), float(code), -(dmin * float(m))));
    } else if constexpr (FMT == GGUF_FMT_IQ4XS || FMT == GGUF_FMT_IQ4NL) {
      // value = scale * codebook[nibble]: byte e % 16 of the group's 16 holds inputs e (low nibble) and 16 + e (high)
      constexpr int kCodebook[16] = {-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113};
      float scale;
      const uint8_t *qs;
      if constexpr (FMT == GGUF_FMT_IQ4XS) {
        const uint32_t high = blk[2] | (blk[3] << 8), ls = ((blk[4u + j / 2u] >> (4u * (j % 2u))) & 15u) | (((high >> (2u * j)) & 3u) << 4);
        scale = half_bits_to_float(blk[0] | (blk[1] << 8)) * float(int(ls) - 32);
        qs = blk + 8u + 16u * j;
      } else {
        scale = half_bits_to_float(blk[18u * j] | (blk[18u * j + 1u] << 8));
        qs = blk + 18u * j + 2u;
      }
      const uint32_t code = e < 16u ? qs[e] & 15u : qs[e - 16u] >> 4;
      return float_to_bf16_bits(scale * float(kCodebook[code]));
    } else if constexpr (FMT == GGUF_FMT_Q80) {
      const uint8_t *group = blk + 34u * j;
      const float d = half_bits_to_float(group[0] | (group[1] << 8));
      return float_to_bf16_bits(d * float(int(int8_t(group[2u + e]))));
    } else {
      const float d = half_bits_to_float(blk[208] | (blk[209] << 8));
      const uint32_t n = k / 128u, r = (k % 128u) / 32u;
      const uint32_t l4 = (blk[64u * n + e + 32u * (r & 1u)] >> (4u * (r >> 1))) & 15u, h2 = (blk[128u + 32u * n + e] >> (2u * r)) & 3u;
      const int q = int(l4 | (h2 << 4)) - 32;
      const float scale = float(int(int8_t(blk[192u + 8u * n + 2u * r + e / 16u])));
      return float_to_bf16_bits(d * scale * float(q));
    }
  }
};

// gguf_embed_<fmt>: out[r][:] = bf16(decode(native row tokens[r])); a token at or past the
// vocabulary gives zeros. Grid (rows, hidden / 256), 64 threads: a thread decodes four values of a super-block.
template <uint32_t FMT>
__global__ __launch_bounds__(64) void gguf_embed(const uint8_t *__restrict__ table, const uint32_t *__restrict__ tokens,
                                                 uint16_t *__restrict__ out, GgufEmbedParams p) {
  const uint32_t row = blockIdx.x, block = blockIdx.y, tid = threadIdx.x;
  const uint32_t token = tokens[row];
  uint16_t *o = out + size_t(row) * p.hidden + size_t(block) * 256u;
  const uint8_t *blk = table + (size_t(token) * (p.hidden / 256u) + block) * EmbedBlock<FMT>::kBytes;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[tid + 64 * i] = token < p.vocabulary ? uint16_t(EmbedBlock<FMT>::bits(blk, tid + 64u * i)) : uint16_t(0);
}
SP_REGISTER_KERNEL("gguf_embed_q4k", &gguf_embed<GGUF_FMT_Q4K>);
SP_REGISTER_KERNEL("gguf_embed_q6k", &gguf_embed<GGUF_FMT_Q6K>);
SP_REGISTER_KERNEL("gguf_embed_q5k", &gguf_embed<GGUF_FMT_Q5K>);
SP_REGISTER_KERNEL("gguf_embed_q80", &gguf_embed<GGUF_FMT_Q80>);
SP_REGISTER_KERNEL("gguf_embed_iq4xs", &gguf_embed<GGUF_FMT_IQ4XS>);
SP_REGISTER_KERNEL("gguf_embed_iq4nl", &gguf_embed<GGUF_FMT_IQ4NL>);

// gguf_embed_norm_<fmt>: the first passes of a step as one: rope_build_tree_tables, gguf_embed and norm_rms_table16 of
// its rows, each the values of its own kernel. Grid (tiles * 16, 2 or 1 without rotary pairs), 256 threads
// or more (the host: a thread an input, up to 1024): a workgroup of y = 0 gathers a row into LDS, stores it, norms it and
// writes its part of the activation table, a thread a vector of eight (zeros past the live rows); one of y = 1 writes the
// row's RoPE tables. Rows of up to kStagedWidth columns. Three launches of a few workgroups each that only waited on one
// another: 3.7 + 4.1 + 5.6 us at 16 rows of 1024 columns, 8.0 together by 256 threads (the gather, the sum and the table are
// one chain of waits), 5.7 by 1024; at 16 rows of 5120 columns 12.9 -> 9.2. And two launches less a step.
template <uint32_t FMT>
__global__ __launch_bounds__(1024) void gguf_embed_norm(const uint8_t *__restrict__ embedding, const uint32_t *__restrict__ tokens,
                                                       const uint16_t *__restrict__ weight, uint16_t *__restrict__ hidden,
                                                       uint16_t *__restrict__ output, uint8_t *__restrict__ table,
                                                       const float *__restrict__ inverse_frequency, const uint32_t *__restrict__ depth,
                                                       float *__restrict__ cosines, float *__restrict__ sines, EmbedNormParams p) {
  __shared__ float scratch[4];
  __shared__ __align__(16) uint16_t rowX[kStagedWidth];
  // a native row in pieces that every format's rows are whole numbers of (a Q6_K block is 210 bytes)
  using Piece = std::conditional_t<FMT == GGUF_FMT_Q6K, uint16_t, uint32_t>;
  constexpr uint32_t kNative = kStagedWidth / 256u * EmbedBlock<FMT>::kBytes / sizeof(Piece), kPieces = (kNative + 1023u) / 1024u;
  __shared__ __align__(16) Piece native[kNative];
  const uint32_t row = blockIdx.x, tid = threadIdx.x, threads = blockDim.x, vectors = p.embed.hidden / 8u;
  const bool live = row < p.embed.rows;
  if (blockIdx.y) {
    if (live)
      for (uint32_t pair = tid; pair < p.rope.pairs; pair += threads) rope_entry(row, pair, inverse_frequency, depth, cosines, sines, p.rope);
    return;
  }
  uint4 norm = make_uint4(0u, 0u, 0u, 0u);
  if (live) {
    const uint32_t token = tokens[row], blocks = p.embed.hidden / 256u;
    const bool inside = token < p.embed.vocabulary;
    // the native row whole, with every load in flight at once (a decode's byte loads from memory wait for one another)
    const uint8_t *source = embedding + size_t(inside ? token : 0u) * blocks * EmbedBlock<FMT>::kBytes;
    const uint32_t pieces = blocks * EmbedBlock<FMT>::kBytes / uint32_t(sizeof(Piece));
    norm = reinterpret_cast<const uint4 *>(weight)[min(tid, vectors - 1u)];
    for (uint32_t first = tid; first < pieces; first += threads * kPieces) {
      uint32_t held[kPieces];
#pragma unroll
      for (uint32_t i = 0; i < kPieces; ++i) {
        Piece piece;
        __builtin_memcpy(&piece, source + min(first + threads * i, pieces - 1u) * sizeof(Piece), sizeof(Piece));
        held[i] = piece;
      }
#pragma unroll
      for (uint32_t i = 0; i < kPieces; ++i) arrived(held[i]);
#pragma unroll
      for (uint32_t i = 0; i < kPieces; ++i)
        if (first + threads * i < pieces) native[first + threads * i] = Piece(held[i]);
    }
    __syncthreads();
    for (uint32_t at = tid; at < p.embed.hidden; at += threads) {
      const uint8_t *block = reinterpret_cast<const uint8_t *>(native) + at / 256u * EmbedBlock<FMT>::kBytes;
      const uint16_t value = inside ? uint16_t(EmbedBlock<FMT>::bits(block, at % 256u)) : uint16_t(0);
      rowX[at] = value;
      hidden[size_t(row) * p.embed.hidden + at] = value;
    }
  }
  __syncthreads();
  const float inverse = live ? rms_inverse(rowX, p.embed.hidden, scratch) : 0.f;
  const uint4 mine = reinterpret_cast<const uint4 *>(rowX)[min(tid, vectors - 1u)];
  write_norm_vectors(mine, norm, rowX, weight, inverse, live, row, output, table, p.embed.hidden, p.tiles);
}
SP_REGISTER_KERNEL("gguf_embed_norm_q4k", &gguf_embed_norm<GGUF_FMT_Q4K>);
SP_REGISTER_KERNEL("gguf_embed_norm_q6k", &gguf_embed_norm<GGUF_FMT_Q6K>);
SP_REGISTER_KERNEL("gguf_embed_norm_q5k", &gguf_embed_norm<GGUF_FMT_Q5K>);
SP_REGISTER_KERNEL("gguf_embed_norm_q80", &gguf_embed_norm<GGUF_FMT_Q80>);
SP_REGISTER_KERNEL("gguf_embed_norm_iq4xs", &gguf_embed_norm<GGUF_FMT_IQ4XS>);
SP_REGISTER_KERNEL("gguf_embed_norm_iq4nl", &gguf_embed_norm<GGUF_FMT_IQ4NL>);

} // namespace splash::kernels
