#pragma once

// A row of the wide table (abi/Gguf.h): what makes it, for the kernels that put it where it goes.
#include "abi/Gguf.h"
#include "abi/Glue.h"
#include "kernels/gguf_records.hpp"

namespace splash::kernels {

typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
__device__ __forceinline__ uint32_t as_word(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
// `Waves` waves a row, whose values stay in registers from their one load to where `put` stores them: thread t of them holds
// the eight inputs of quarter t % 4 of groups t / 4, 16 Waves + t / 4, ... in `Held` pieces. put(line, g, kq, entry): the
// row's place among the sixteen of line `line` of its tile (a line: one quarter of one operand, sixteen rows of 16 bytes).
// Returns the row's scale.
// (The operands, the parts of their sums and the scale are the same bits whatever Waves is; a norm's sum of squares is added
// over four waves.)
template <uint32_t Waves> constexpr uint32_t kWidePiece = 16u * Waves;   // groups of 32 inputs a piece
// A thread's part of a row (or of a norm's weights): piece i holds inputs 4 kq .. + 3, then 16 + 4 kq .. + 3 of group
// 16 Waves i + t / 4, zeros of a row that is not there.
template <uint32_t Held, uint32_t Waves>
__device__ __forceinline__ void wide_row_load(uint4 (&v)[Held], const uint16_t *from, uint32_t inputSize, bool live) {
  const uint32_t tid = threadIdx.x % (64u * Waves), kq = tid & 3u, groups = inputSize / 32u, held = (groups + kWidePiece<Waves> - 1u) / kWidePiece<Waves>;
#pragma unroll
  for (uint32_t i = 0; i < Held; ++i)
    if (i < held) {
      const uint32_t g = kWidePiece<Waves> * i + (tid >> 2);
      v[i] = make_uint4(0u, 0u, 0u, 0u);
      if (!live || g >= groups) continue;
      const uint2 a = *reinterpret_cast<const uint2 *>(from + 32u * g + 4u * kq), b = *reinterpret_cast<const uint2 *>(from + 32u * g + 16u + 4u * kq);
      v[i] = make_uint4(a.x, a.y, b.x, b.y);
    }
}
// The row's inverse RMS, over the four waves that hold it.
template <uint32_t Held>
__device__ __forceinline__ float wide_row_inverse(const uint4 (&v)[Held], uint32_t inputSize, float *scratch) {
  const uint32_t held = (inputSize / 32u + kWidePiece<4> - 1u) / kWidePiece<4>;
  float sum = 0.f;
#pragma unroll
  for (uint32_t i = 0; i < Held; ++i)
    if (i < held) {
      const uint32_t words[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float low = bf16_bits_to_float(words[e] & 0xFFFFu), high = bf16_bits_to_float(words[e] >> 16);
        sum += low * low;
        sum += high * high;
      }
    }
  sum = wave_sum(sum);
  if ((threadIdx.x & 63u) == 0) scratch[threadIdx.x >> 6] = sum;
  __syncthreads();
  return 1.0f / sqrtf((((scratch[0] + scratch[1]) + scratch[2]) + scratch[3]) / float(inputSize) + SPLASH_RMS_EPSILON);
}
// bf16((x * inverse) * weight)
template <uint32_t Held>
__device__ __forceinline__ void wide_row_norm(uint4 (&out)[Held], const uint4 (&v)[Held], const uint4 (&w)[Held], float inverse, uint32_t inputSize) {
  const uint32_t held = (inputSize / 32u + kWidePiece<4> - 1u) / kWidePiece<4>;
#pragma unroll
  for (uint32_t i = 0; i < Held; ++i)
    if (i < held) {
      const uint32_t words[4] = {v[i].x, v[i].y, v[i].z, v[i].w}, weights[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
      uint32_t normed[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t low = float_to_bf16_bits((bf16_bits_to_float(words[e] & 0xFFFFu) * inverse) * bf16_bits_to_float(weights[e] & 0xFFFFu));
        const uint32_t high = float_to_bf16_bits((bf16_bits_to_float(words[e] >> 16) * inverse) * bf16_bits_to_float(weights[e] >> 16));
        normed[e] = low | (high << 16);
      }
      out[i] = make_uint4(normed[0], normed[1], normed[2], normed[3]);
    }
}
// The row's entries of what the threads hold. (scratch: four floats that no earlier row of the workgroup still reads)
template <uint32_t Held, uint32_t Waves, class Put>
__device__ __forceinline__ float wide_row_entries(const uint4 (&v)[Held], uint32_t inputSize, float *scratch, Put &&put) {
  constexpr uint32_t kPiece = kWidePiece<Waves>;
  const uint32_t tid = threadIdx.x % (64u * Waves), lane = tid & 63u, wave = tid >> 6;
  const uint32_t kq = tid & 3u, groups = inputSize / 32u, held = (groups + kPiece - 1u) / kPiece;
  uint32_t largest = 0;
#pragma unroll
  for (uint32_t i = 0; i < Held; ++i)
    if (i < held) {
      const uint32_t words[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t low = words[e] & 0x7FFFu, high = (words[e] >> 16) & 0x7FFFu;
        if (low < 0x7F80u) largest = max(largest, low);   // (an infinity or NaN stays what it is)
        if (high < 0x7F80u) largest = max(largest, high);
      }
    }
  largest = wave_max(largest);
  if constexpr (Waves > 1u) {
    if (lane == 0) scratch[wave] = __uint_as_float(largest);
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 4; ++w) largest = max(largest, __float_as_uint(scratch[w]));
  }
  // 2^e, e = 14 - the exponent of the largest magnitude (a row of zeros or of subnormals: the largest 2^e there is)
  const uint32_t exponent = max(largest >> 7, 15u);
  const float scale = __uint_as_float((141u + 127u - exponent) << 23), inverseScale = __uint_as_float((exponent - 14u) << 23);
#pragma unroll
  for (uint32_t i = 0; i < Held; ++i)
    if (i < held) {
      const uint32_t g = kPiece * i + (tid >> 2);
      const uint32_t words[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
      float f[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f[2 * e] = bf16_bits_to_float(words[e] & 0xFFFFu) * scale;
        f[2 * e + 1] = bf16_bits_to_float(words[e] >> 16) * scale;
      }
      // inputs 4 kq + {0, 2, 1, 3} of each half group
      auto pair = [](float a, float b) { return f16x2{_Float16(a), _Float16(b)}; };
      const f16x2 operand[4] = {pair(f[0], f[2]), pair(f[1], f[3]), pair(f[4], f[6]), pair(f[5], f[7])};
      if (g < groups)
        put(((g >> 3) * GGUF_WIDE_OPERANDS + (g & 7u)) * 4u + kq, g & 7u, kq,
            make_uint4(as_word(operand[0]), as_word(operand[1]), as_word(operand[2]), as_word(operand[3])));
      // the group's sum of what the operands hold, in three fp16 parts
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) s += float(operand[e].x) + float(operand[e].y);
      s += lane_xor<1>(s);
      s += lane_xor<2>(s);
      s *= 0.03125f;
      const float first = float(_Float16(s)), second = float(_Float16(s - first)), third = float(_Float16((s - first) - second));
      const float mine = kq == 0u ? first : kq == 1u ? second : kq == 2u ? third : 0.f;
      // element g % 8 of the super-block's operand: the halves of eight threads into one 16-byte store
      const uint32_t part = as_word(f16x2{_Float16(mine), _Float16(0.f)}) & 0xFFFFu;
      const uint32_t two = part | (lane_down<4>(part) << 16);
      const uint32_t b = lane_down<8>(two), c = uint32_t(__shfl_down(int(two), 16, 64)), d = uint32_t(__shfl_down(int(two), 24, 64));
      if ((g & 7u) == 0 && g < groups) put(((g >> 3) * GGUF_WIDE_OPERANDS + 8u) * 4u + kq, 8u, kq, make_uint4(two, b, c, d));
    }
  return inverseScale;
}
template <bool Norm, uint32_t Held, uint32_t Waves, class Put>
__device__ __forceinline__ float wide_table_row(const uint16_t *__restrict__ input, const uint16_t *__restrict__ weight, const GgufWideTableParams &p,
                                                const uint32_t source, Put &&put) {
  static_assert(Waves == 4u || (Waves == 1u && !Norm), "a row of one wave has no other wave's sums to add");
  __shared__ float scratch[8];
  const bool live = source < p.rows;
  uint4 v[Held];
  wide_row_load<Held, Waves>(v, input + size_t(live ? source : 0u) * p.input_size, p.input_size, live);
  if constexpr (Norm) {
    uint4 w[Held];
    wide_row_load<Held, Waves>(w, weight, p.input_size, live);
    wide_row_norm(v, v, w, wide_row_inverse(v, p.input_size, scratch), p.input_size);
  }
  return wide_row_entries<Held, Waves>(v, p.input_size, scratch + 4, put);
}
__device__ __forceinline__ float *wide_scales_of(uint8_t *table, const GgufWideTableParams &p) {
  return reinterpret_cast<float *>(table + gguf_wide_scales_offset(p.input_size, p.tiles));
}
__device__ __forceinline__ uint32_t wide_table_row_of(uint32_t block) {
  const uint32_t die = block % 8u, slot = block / 8u;
  return (slot / 8u * 8u + die) * 8u + slot % 8u;
}

} // namespace splash::kernels
