// Block-causal attention of a verify block over the paged INT8 KV cache, for gfx950 (the
// reference's kernels/shared/attention_qkv.metal, paged_attention.metal, kv_path_commit.metal and
// common/paged_attention_tile.h, attention_qkv_prepare.h, attention_store.h).
//
//   attention_q8_qkv_d<D>     per (head, row, sequence): RMS-norm q and k, partial RoPE, stage the
//                             query rows, quantize k and v into the row's page slot.
//   attention_q8_split_d<D>_g<G>  per (KV head, history split, sequence): flash-decoding page loop
//                             over the split's 64-token steps for all 16 G fused rows of the head.
//   attention_q8_few_d<D>_g<G>_t<T>  the same for blocks of up to eight rows, a wave a split.
//   attention_reduce_d<D>     per (query head, row, sequence): merge the splits in split order.
//   attention_q8_commit_d<D>  per (KV head, sequence): move the retained path's slots to their depths.
//
// The page loop keeps the reference's rules (paged_attention_tile.h:179-285): score =
// (q . k_codes) key_scale / sqrt(D), computed on the stored integer codes; online softmax per step;
// P is folded with value_scale before the P.V product, which also runs on the stored codes. Both
// products are fp16 MFMAs on exact integer operands: a stored code c becomes the fp16 number
// 1152 + c by one byte permute (0x6400 | (c ^ 0x80), no conversion instruction), and the constant
// 1152 is removed exactly afterwards with the row's sum of q (scores) and of P (outputs), the latter
// from one more MFMA against a tile of ones. Scores are kept transposed (tokens x rows) so that a
// lane owns one fused row from the first MFMA to the last: row maxima, sums and rescales never
// cross lanes except over the four lanes that share a row.
#include "abi/Gguf.h"
#include "abi/PagedAttention.h"
#include "backend/KernelRegistry.hpp"
#include "kernels/acceptance.hpp"
#include "kernels/gguf_records.hpp"   // buffer resources
#include <type_traits>

namespace splash::kernels {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;

constexpr float kCodeOffset = 1152.0f;  // fp16(0x6400 | u) = 1024 + u, u = code + 128
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kPScale = 1024.0f;  // P is carried times 2^10 so that small weights stay normal fp16

// Bytes b0..b3 of x as two registers of fp16 numbers 1024 + b: [b0, b1] and [b2, b3].
__device__ __forceinline__ uint2 bytes_to_f16(uint32_t x) {
  return make_uint2(__builtin_amdgcn_perm(0x64646464u, x, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, x, 0x04030402u));
}

template <int N> __device__ __forceinline__ float block_sum(float v, float *scratch, uint32_t tid) {
  v = wave_sum(v);
  if constexpr (N > 64) {
    if ((tid & 63u) == 0) scratch[tid >> 6] = v;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < N / 64; ++w) total += scratch[w];
    __syncthreads();
    return total;
  }
  return v;
}
template <int N> __device__ __forceinline__ float block_max(float v, float *scratch, uint32_t tid) {
  v = wave_max(v);
  if constexpr (N > 64) {
    if ((tid & 63u) == 0) scratch[tid >> 6] = v;
    __syncthreads();
    float total = scratch[0];
#pragma unroll
    for (int w = 1; w < N / 64; ++w) total = fmaxf(total, scratch[w]);
    __syncthreads();
    return total;
  }
  return v;
}

// Block z of a dispatch. A prompt chunk's kernels (Chunk) work it out from the chunk's one sequence; a step's read its
// sequence at once, without a test of chunk_rows before it.
template <bool Chunk> __device__ __forceinline__ AttentionSequence block_sequence(const AttentionParams &p, uint32_t z) {
  if constexpr (Chunk) return attention_sequence(p, z);
  else return p.sequence[z];
}

// The page of logical page `index` of a sequence.
__device__ __forceinline__ uint8_t *page_of(uint8_t *pool, const uint64_t *page_table, const AttentionSequence &seq,
                                            uint64_t page_bytes, uint32_t index) {
  return pool + page_table[seq.table_first + index] * page_bytes;
}

// attention_store.h:52-85: scale = max / 127, code = clamp(rint(v 127 / max)); the scale is stored fp16.
__device__ __forceinline__ int8_t cache_code(float v, float maximum) {
  if (maximum == 0.0f) return 0;
  const int q = int(rintf(v * 127.0f / maximum));
  return int8_t(q < -127 ? -127 : q > 127 ? 127 : q);
}
__device__ __forceinline__ void store_cache_scales(uint8_t *page, uint32_t kv_heads, uint32_t D, uint32_t head, uint32_t token, float keyMax,
                                                   float valueMax) {
  uint16_t *ks = reinterpret_cast<uint16_t *>(page + attention_page_key_scales_offset(kv_heads, D));
  uint16_t *vs = reinterpret_cast<uint16_t *>(page + attention_page_value_scales_offset(kv_heads, D));
  ks[attention_scale_index(head, token)] = uint16_t(float_to_half_bits(keyMax == 0.0f ? 0.0f : keyMax / 127.0f));
  vs[attention_scale_index(head, token)] = uint16_t(float_to_half_bits(valueMax == 0.0f ? 0.0f : valueMax / 127.0f));
}

// ---------------------------------------------------------------------------------------------
// attention_q8_qkv: grid (q_heads + kv_heads, 16, sequences), D threads.
// Staged queries: fp16 [sequence][kv head][group head][16 rows][D] (rows past the block zero) and
// their fp32 sums [sequence][kv head][group head][16].
// ---------------------------------------------------------------------------------------------
template <int D, bool Chunk>
__global__ __launch_bounds__(D) void attention_q8_qkv(const uint16_t *__restrict__ qkv, const uint16_t *__restrict__ q_norm,
                                                      const uint16_t *__restrict__ k_norm, const float *__restrict__ rope_cos,
                                                      const float *__restrict__ rope_sin, _Float16 *__restrict__ queries,
                                                      float *__restrict__ qsums, const uint64_t *__restrict__ page_table,
                                                      uint8_t *__restrict__ pool, AttentionParams p) {
  __shared__ float scratch[4];
  __shared__ float normalized[D];
  const uint32_t tid = threadIdx.x, head = blockIdx.x, row = blockIdx.y, z = blockIdx.z;
  const AttentionSequence seq = block_sequence<Chunk>(p, z);
  const bool query = head < p.q_heads;
  const uint32_t group = p.q_heads / p.kv_heads;
  if (row >= seq.rows) {
    if (query) {
      const uint32_t kv = head / group, g = head % group;
      const size_t at = ((size_t(z) * p.kv_heads + kv) * group + g) * 16u + row;
      if (!Chunk && p.int8_queries) reinterpret_cast<int8_t *>(queries)[at * D + tid] = 0;
      else queries[at * D + tid] = _Float16(0.f);
      if (tid == 0) qsums[at] = 0.f;
    }
    return;
  }
  const uint32_t index = query ? head : head - p.q_heads;
  const size_t packed = size_t(seq.first_row) + row;
  // A gated layer's row holds each query head's queries, then its gate (attention_gate.h:27-31).
  const uint32_t queryStride = p.gated ? 2u * D : uint32_t(D);
  const uint16_t *source = qkv + packed * p.qkv_stride + (query ? index * queryStride : p.q_heads * queryStride + index * D);
  const float element = bf16_bits_to_float(source[tid]);
  float result = element;
  if (p.normalize) {
    // attention_qkv_prepare.h:59-66: inv = rsqrt(sum x^2 / D + 1e-6); n = bf16(x inv w)
    const float total = block_sum<D>(element * element, scratch, tid);
    const float inverse = 1.0f / sqrtf(total / float(D) + 1e-6f);  // correctly rounded, as the CPU oracle's
    result = round_bf16(element * inverse * bf16_bits_to_float((query ? q_norm : k_norm)[tid]));
  }
  if (p.rotary_pairs) {
    normalized[tid] = result;
    __syncthreads();
    if (tid < 2 * p.rotary_pairs) {
      const uint32_t pair = tid % p.rotary_pairs;
      const float first = normalized[pair], second = normalized[pair + p.rotary_pairs];
      const float cosine = rope_cos[packed * p.rotary_pairs + pair], sine = rope_sin[packed * p.rotary_pairs + pair];
      result = tid < p.rotary_pairs ? round_bf16(first * cosine - second * sine) : round_bf16(second * cosine + first * sine);
    }
  }
  if (query) {
    const uint32_t kv = index / group, g = index % group;
    const size_t at = ((size_t(z) * p.kv_heads + kv) * group + g) * 16u + row;
    if (!Chunk && p.int8_queries) {   // (a prompt chunk's queries are fp16: planPrompt refuses others)
      // common/int8_activations.h:22-28: code = clamp(rint(x (127 / m))), the quotient rounded first; scale = m / 127; a
      // head at or below 2^-100 codes as zeros with scale 0; one that is not finite takes a NaN scale. The codes lie
      // where the fp16 queries would, one byte a dimension, and the scale in the sums' slot.
      const uint32_t bits = __builtin_bit_cast(uint32_t, result);
      const float notFinite = block_max<D>((bits & 0x7F800000u) == 0x7F800000u ? 1.f : 0.f, scratch, tid);
      const float largest = block_max<D>(fabsf(result), scratch, tid);
      const bool coded = largest > 0x1p-100f;
      const float inverse = coded ? 127.0f / largest : 0.0f;
      const float code = fminf(fmaxf(rintf(result * inverse), -127.0f), 127.0f);
      reinterpret_cast<int8_t *>(queries)[at * D + tid] = notFinite != 0.f ? int8_t(0) : int8_t(code);
      if (tid == 0) qsums[at] = notFinite != 0.f ? __builtin_bit_cast(float, 0x7FC00000u) : coded ? largest / 127.0f : 0.0f;
      return;
    }
    const _Float16 staged = _Float16(result);
    queries[at * D + tid] = staged;
    const float sum = block_sum<D>(float(staged), scratch, tid);
    if (tid == 0) qsums[at] = sum;
    return;
  }
  const float value = bf16_bits_to_float(source[p.kv_heads * D + tid]);
  const float keyMax = block_max<D>(fabsf(result), scratch, tid), valueMax = block_max<D>(fabsf(value), scratch, tid);
  const uint32_t slot = seq.committed + row, token = slot % ATTENTION_PAGE_TOKENS;
  uint8_t *page = page_of(pool, page_table, seq, p.page_bytes, slot / ATTENTION_PAGE_TOKENS);
  reinterpret_cast<int8_t *>(page)[attention_key_index(index, token, tid, D)] = cache_code(result, keyMax);
  reinterpret_cast<int8_t *>(page + attention_page_values_offset(p.kv_heads, D))[attention_value_index(index, token, tid, D)] =
      cache_code(value, valueMax);
  if (tid == 0) store_cache_scales(page, p.kv_heads, D, index, token, keyMax, valueMax);
}
SP_REGISTER_KERNEL("attention_q8_qkv_d128", (&attention_q8_qkv<128, false>));
SP_REGISTER_KERNEL("attention_q8_qkv_d64", (&attention_q8_qkv<64, false>));
SP_REGISTER_KERNEL("attention_q8_qkv_chunk_d128", (&attention_q8_qkv<128, true>));
SP_REGISTER_KERNEL("attention_q8_qkv_chunk_d64", (&attention_q8_qkv<64, true>));

// The same for a prompt chunk's many blocks: grid (q_heads + kv_heads, sequences), a workgroup a head's whole block, each
// wavefront four of its rows with their loads in flight together and lane l elements l and l + 64 of each. No barrier, and
// sums and maxima in attention_q8_qkv's order (each 64 elements by a wavefront, then the halves), so every byte is the same.
// A workgroup a row is bound by how fast workgroups start (147456 of them for 2048 rows of 64 / 8 heads): 114 us there, 45 at
// 777 rows, against 76 and 36 here. Four rows one after the other take 14.5 us however few the blocks are.
template <int D>
__device__ __forceinline__ void qkv_rows_of_head(const uint32_t head, const uint16_t *__restrict__ qkv, const uint16_t *__restrict__ q_norm,
                                                 const uint16_t *__restrict__ k_norm, const float *__restrict__ rope_cos,
                                                 const float *__restrict__ rope_sin, _Float16 *__restrict__ queries, float *__restrict__ qsums,
                                                 const uint64_t *__restrict__ page_table, uint8_t *__restrict__ pool, const AttentionParams &p) {
  constexpr uint32_t E = D / 64, kRows = 4;
  __shared__ float normalized[4][D];
  const uint32_t l = threadIdx.x & 63u, wave = threadIdx.x >> 6, z = blockIdx.y;
  const AttentionSequence seq = block_sequence<true>(p, z);
  const bool query = head < p.q_heads;
  const uint32_t group = p.q_heads / p.kv_heads, index = query ? head : head - p.q_heads, pairs = p.rotary_pairs;
  const uint32_t queryStride = p.gated ? 2u * D : uint32_t(D);
  const uint32_t offset = query ? index * queryStride : p.q_heads * queryStride + index * D;
  auto sumOf = [](const float (&v)[E]) __attribute__((always_inline)) {
    float total = wave_sum(v[0]);
    if constexpr (E > 1) {
      total = 0.f + total;
#pragma unroll
      for (uint32_t e = 1; e < E; ++e) total += wave_sum(v[e]);
    }
    return total;
  };
  auto maximumOf = [](const float (&v)[E]) __attribute__((always_inline)) {
    if constexpr (E == 1) return wave_max(v[0]);
    auto first = [](float m) { return __uint_as_float(uint32_t(__builtin_amdgcn_readfirstlane(int(__float_as_uint(m))))); };
    float most = first(wave_max(v[0]));
#pragma unroll
    for (uint32_t e = 1; e < E; ++e) most = fmaxf(most, first(wave_max(v[e])));
    return most;
  };

  float element[kRows][E], value[kRows][E], cosine[kRows][E], sine[kRows][E], weight[E];
#pragma unroll
  for (uint32_t j = 0; j < kRows; ++j) {
    const uint32_t row = 4u * wave + j;
    const bool live = row < seq.rows;
    const size_t packed = size_t(seq.first_row) + row;
    const uint16_t *source = qkv + packed * p.qkv_stride + offset;
#pragma unroll
    for (uint32_t e = 0; e < E; ++e) {
      const uint32_t d = l + 64u * e;
      const bool turns = live && d < 2u * pairs;
      element[j][e] = live ? bf16_bits_to_float(source[d]) : 0.f;
      value[j][e] = live && !query ? bf16_bits_to_float(source[p.kv_heads * D + d]) : 0.f;
      const uint32_t pair = d < pairs ? d : d - pairs;
      cosine[j][e] = turns ? rope_cos[packed * pairs + pair] : 0.f;
      sine[j][e] = turns ? rope_sin[packed * pairs + pair] : 0.f;
    }
  }
#pragma unroll
  for (uint32_t e = 0; e < E; ++e) weight[e] = p.normalize ? bf16_bits_to_float((query ? q_norm : k_norm)[l + 64u * e]) : 1.f;

#pragma unroll
  for (uint32_t j = 0; j < kRows; ++j) {
    const uint32_t row = 4u * wave + j;
    const size_t at = ((size_t(z) * p.kv_heads + index / group) * group + index % group) * 16u + row;   // (a query head's)
    if (row >= seq.rows) {
      if (query) {
#pragma unroll
        for (uint32_t e = 0; e < E; ++e) queries[at * D + l + 64u * e] = _Float16(0.f);
        if (l == 0) qsums[at] = 0.f;
      }
      continue;
    }
    float result[E];
#pragma unroll
    for (uint32_t e = 0; e < E; ++e) result[e] = element[j][e];
    if (p.normalize) {
      float squares[E];
#pragma unroll
      for (uint32_t e = 0; e < E; ++e) squares[e] = element[j][e] * element[j][e];
      const float inverse = 1.0f / sqrtf(sumOf(squares) / float(D) + 1e-6f);
#pragma unroll
      for (uint32_t e = 0; e < E; ++e) result[e] = round_bf16(element[j][e] * inverse * weight[e]);
    }
    if (pairs) {
      wave_lds_fence();
#pragma unroll
      for (uint32_t e = 0; e < E; ++e) normalized[wave][l + 64u * e] = result[e];
      wave_lds_fence();
#pragma unroll
      for (uint32_t e = 0; e < E; ++e) {
        const uint32_t d = l + 64u * e;
        if (d < 2u * pairs) {
          const float first = normalized[wave][d < pairs ? d : d - pairs], second = normalized[wave][d < pairs ? d + pairs : d];
          result[e] = d < pairs ? round_bf16(first * cosine[j][e] - second * sine[j][e]) : round_bf16(second * cosine[j][e] + first * sine[j][e]);
        }
      }
    }
    if (query) {
      float staged[E];
#pragma unroll
      for (uint32_t e = 0; e < E; ++e) {
        const _Float16 half = _Float16(result[e]);
        queries[at * D + l + 64u * e] = half;
        staged[e] = float(half);
      }
      const float sum = sumOf(staged);
      if (l == 0) qsums[at] = sum;
    } else {
      float keyMagnitude[E], valueMagnitude[E];
#pragma unroll
      for (uint32_t e = 0; e < E; ++e) {
        keyMagnitude[e] = fabsf(result[e]);
        valueMagnitude[e] = fabsf(value[j][e]);
      }
      const float keyMax = maximumOf(keyMagnitude), valueMax = maximumOf(valueMagnitude);
      const uint32_t slot = seq.committed + row, token = slot % ATTENTION_PAGE_TOKENS;
      uint8_t *page = page_of(pool, page_table, seq, p.page_bytes, slot / ATTENTION_PAGE_TOKENS);
#pragma unroll
      for (uint32_t e = 0; e < E; ++e) {
        const uint32_t d = l + 64u * e;
        reinterpret_cast<int8_t *>(page)[attention_key_index(index, token, d, D)] = cache_code(result[e], keyMax);
        reinterpret_cast<int8_t *>(page + attention_page_values_offset(p.kv_heads, D))[attention_value_index(index, token, d, D)] =
            cache_code(value[j][e], valueMax);
      }
      if (l == 0) store_cache_scales(page, p.kv_heads, D, index, token, keyMax, valueMax);
    }
  }
}
template <int D>
__global__ __launch_bounds__(256) void attention_q8_qkv_rows(const uint16_t *__restrict__ qkv, const uint16_t *__restrict__ q_norm,
                                                            const uint16_t *__restrict__ k_norm, const float *__restrict__ rope_cos,
                                                            const float *__restrict__ rope_sin, _Float16 *__restrict__ queries,
                                                            float *__restrict__ qsums, const uint64_t *__restrict__ page_table,
                                                            uint8_t *__restrict__ pool, AttentionParams p) {
  qkv_rows_of_head<D>(blockIdx.x, qkv, q_norm, k_norm, rope_cos, rope_sin, queries, qsums, page_table, pool, p);
}
SP_REGISTER_KERNEL("attention_q8_qkv_rows_d128", &attention_q8_qkv_rows<128>);
SP_REGISTER_KERNEL("attention_q8_qkv_rows_d64", &attention_q8_qkv_rows<64>);

// The sum that a wavefront's butterfly over 64 elements gives, of eight lanes that hold eight elements each: lane bits 0, 1 and
// 2 are the elements' bits 5, 4 and 3, so that the lanes are added first, and what a lane holds last. In all eight lanes.
__device__ __forceinline__ float sum_of_eights(const float (&v)[8]) {
  float s[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) s[i] = dpp_add<kRowHalfMirror>(dpp_add<kQuadSwap2>(dpp_add<kQuadSwap1>(v[i])));
  return ((s[0] + s[4]) + (s[2] + s[6])) + ((s[1] + s[5]) + (s[3] + s[7]));
}
// The same where a row's vectors are whole (rotary pairs a multiple of eight, sixteen-byte rows, weights and tables): a query
// head's row is D / 8 lanes of eight elements, so that a sum is three steps between lanes for several rows at once, loads and
// stores are sixteen bytes, and a row's cosines and sines serve kHeads heads. Grid (groups of query heads, then the key heads,
// sequences): a key head's workgroup is attention_q8_qkv_rows'. Every byte is the same. A row a wave spent its time in its sums'
// steps, a square root and a division for 128 values: 2048 rows of 64 / 8 heads 68.4 us so and 42.8 here, 777 33.0 and 20.7.
template <int D>
__global__ __launch_bounds__(256) void attention_q8_qkv_vectors(const uint16_t *__restrict__ qkv, const uint16_t *__restrict__ q_norm,
                                                               const uint16_t *__restrict__ k_norm, const float *__restrict__ rope_cos,
                                                               const float *__restrict__ rope_sin, _Float16 *__restrict__ queries,
                                                               float *__restrict__ qsums, const uint64_t *__restrict__ page_table,
                                                               uint8_t *__restrict__ pool, AttentionParams p) {
  constexpr uint32_t kLanes = D / 8, kRows = 64 / kLanes, kWaves = 16 / kRows, kHeads = 4, kGroup = kHeads * (4 / kWaves);
  static_assert(kGroup == ATTENTION_VECTOR_HEADS(D));
  const uint32_t groups = (p.q_heads + kGroup - 1u) / kGroup;
  if (blockIdx.x >= groups) {
    qkv_rows_of_head<D>(p.q_heads + blockIdx.x - groups, qkv, q_norm, k_norm, rope_cos, rope_sin, queries, qsums, page_table, pool, p);
    return;
  }
  __shared__ __align__(16) float normalized[4][kRows][D];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, z = blockIdx.y, k = lane % kLanes;
  const AttentionSequence seq = block_sequence<true>(p, z);
  const uint32_t row = wave % kWaves * kRows + lane / kLanes, firstHead = blockIdx.x * kGroup + wave / kWaves * kHeads, pairs = p.rotary_pairs;
  const bool live = row < seq.rows;
  const size_t packed = size_t(seq.first_row) + row;
  const uint32_t d = 64u * (k >> 3) + 32u * (k & 1u) + 8u * (k & 2u) + 2u * (k & 4u), queryStride = p.gated ? 2u * D : uint32_t(D);
  const bool turns = d < 2u * pairs;
  const uint32_t pair = d < pairs ? d : d - pairs;
  auto vector = [](const uint16_t *from) { return *reinterpret_cast<const uint4 *>(from); };
  uint4 held[kHeads], weights = make_uint4(0u, 0u, 0u, 0u);
  float4 cosine[2] = {}, sine[2] = {};
#pragma unroll
  for (uint32_t h = 0; h < kHeads; ++h)
    held[h] = live && firstHead + h < p.q_heads ? vector(qkv + packed * p.qkv_stride + (firstHead + h) * queryStride + d) : weights;
  if (live && turns) {
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
      cosine[i] = *reinterpret_cast<const float4 *>(rope_cos + packed * pairs + pair + 4u * i);
      sine[i] = *reinterpret_cast<const float4 *>(rope_sin + packed * pairs + pair + 4u * i);
    }
  }
  if (p.normalize) weights = vector(q_norm + d);
  auto each = [](const uint4 &v, float (&out)[8]) {
    const uint32_t words[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      out[2 * i] = bf16_bits_to_float(words[i] & 0xFFFFu);
      out[2 * i + 1] = bf16_bits_to_float(words[i] >> 16);
    }
  };
  auto sumOf = [&](const float (&v)[8]) {
    const float mine = sum_of_eights(v);
    if constexpr (kLanes == 8) return mine;
    const float other = lane_xor<8>(mine), first = k < 8u ? mine : other, second = k < 8u ? other : mine;
    return (0.f + first) + second;
  };
  const float cosines[8] = {cosine[0].x, cosine[0].y, cosine[0].z, cosine[0].w, cosine[1].x, cosine[1].y, cosine[1].z, cosine[1].w};
  const float sines[8] = {sine[0].x, sine[0].y, sine[0].z, sine[0].w, sine[1].x, sine[1].y, sine[1].z, sine[1].w};
  float weight[8], *mine = normalized[wave][lane / kLanes];
  each(weights, weight);
#pragma unroll
  for (uint32_t h = 0; h < kHeads; ++h) {
    const uint32_t head = firstHead + h, group = p.q_heads / p.kv_heads;
    if (head >= p.q_heads) break;
    float result[8];
    each(held[h], result);
    if (p.normalize) {
      float squares[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) squares[i] = result[i] * result[i];
      const float inverse = 1.0f / sqrtf(sumOf(squares) / float(D) + 1e-6f);
#pragma unroll
      for (int i = 0; i < 8; ++i) result[i] = round_bf16(result[i] * inverse * weight[i]);
    }
    if (pairs) {
      wave_lds_fence();
      reinterpret_cast<float4 *>(mine + d)[0] = make_float4(result[0], result[1], result[2], result[3]);
      reinterpret_cast<float4 *>(mine + d)[1] = make_float4(result[4], result[5], result[6], result[7]);
      wave_lds_fence();
      if (turns) {
        const float4 *partner = reinterpret_cast<const float4 *>(mine + (d < pairs ? d + pairs : pair));
        const float4 a = partner[0], b = partner[1];
        const float others[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 8; ++i)
          result[i] = d < pairs ? round_bf16(result[i] * cosines[i] - others[i] * sines[i]) : round_bf16(result[i] * cosines[i] + others[i] * sines[i]);
      }
    }
    f16x8 halves;
    float staged[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      halves[i] = live ? _Float16(result[i]) : _Float16(0.f);
      staged[i] = float(halves[i]);
    }
    const float sum = sumOf(staged);
    const size_t at = ((size_t(z) * p.kv_heads + head / group) * group + head % group) * 16u + row;
    *reinterpret_cast<f16x8 *>(queries + at * D + d) = halves;
    if (k == 0) qsums[at] = live ? sum : 0.f;
  }
}
SP_REGISTER_KERNEL("attention_q8_qkv_vectors_d128", &attention_q8_qkv_vectors<128>);
SP_REGISTER_KERNEL("attention_q8_qkv_vectors_d64", &attention_q8_qkv_vectors<64>);

// ---------------------------------------------------------------------------------------------
// attention_q8_split: grid (kv_heads, splits, sequences), 256 threads.
// Partials: O fp32 [sequence][kv head][split][16 G fused rows][D], (max, sum) fp32 pairs
// [sequence][kv head][split][16 G]; the max is in the log2 domain of the scaled scores.
// ---------------------------------------------------------------------------------------------
// I8: the queries are INT8 codes with a scale a fused row (attention_q8_qkv staged them so): the score product is one
// v_mfma_i32_16x16x64_i8 per 64 dimensions on the keys' stored bytes, which pass through LDS as they are (no widening,
// no offset to remove), and a row's scale multiplies its scores after the product.
typedef __attribute__((ext_vector_type(4))) int i32x4;
// Whole: the workgroup's split is the block's whole history, and its rows leave finished (to `out`, gated by `packed`'s
// gates where the layer has them) instead of as partials.
template <int D, int G, bool I8, bool Whole, bool Chunk>
__device__ __forceinline__ void attention_split(const _Float16 *__restrict__ queries, const float *__restrict__ qsums,
                                                const AttentionTreeRow *__restrict__ tree, const uint64_t *__restrict__ page_table,
                                                uint8_t *__restrict__ pool, _Float16 *__restrict__ partialO, float *__restrict__ partialML,
                                                uint16_t *__restrict__ out, const uint16_t *__restrict__ packed, const AttentionParams &p,
                                                const uint32_t h, const uint32_t split, const uint32_t z) {
  constexpr int kStep = 64, JD = D / 32, DT = D / 16;
  constexpr int kTiles = (G + 3) / 4;  // fused-row tiles (one query head's 16 rows each) per wave
  constexpr int kKeyVectors = kStep * D / 16 / 256, kValueVectors = kKeyVectors;
  static_assert(kKeyVectors >= 1, "a step's keys fill the workgroup's loads");
  // keys: fp16 numbers 1152 + code, or (I8) the stored bytes, a token's row padded by 16 bytes either way
  constexpr int kKeyRow = I8 ? (D + 16) / 2 : D + 8;  // in fp16 units
  __shared__ __align__(16) _Float16 ldsK[2][kStep][kKeyRow];
  __shared__ __align__(16) _Float16 ldsV[2][D][kStep + 8];
  __shared__ __align__(16) float ldsKS[2][kStep], ldsVS[2][kStep];

  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, row = lane & 15u, kq = lane >> 4;
  const AttentionSequence seq = block_sequence<Chunk>(p, z);
  const uint32_t total = seq.committed + seq.rows;
  // The sequence's own splits: ceil(steps / steps_per_split) of them; later grid rows are empty.
  static_assert(kStep == int(ATTENTION_STEP_TOKENS) && ATTENTION_PAGE_TOKENS % ATTENTION_STEP_TOKENS == 0, "a page holds whole steps");
  const uint32_t span = uint32_t(seq.steps_per_split) * ATTENTION_STEP_TOKENS;
  const uint32_t first = min(total, split * span), last = min(total, (split + 1) * span);
  const uint32_t steps = first < last ? (last - first + kStep - 1) / kStep : 0;
  const float scale2 = kLog2e / sqrtf(float(D));

  // This wave's query rows as MFMA operands, their sums and their rows' visibility masks.
  constexpr int JQ = D / 64;  // INT8 products of 64 dimensions
  f16x8 q[I8 ? 1 : kTiles][I8 ? 1 : JD];
  i32x4 q8[I8 ? kTiles : 1][I8 ? JQ : 1];
  float qsum[kTiles];  // fp16 queries: the code offset's share of a score; INT8 queries: the row's scale
  bool owns[kTiles];
#pragma unroll
  for (int k = 0; k < kTiles; ++k) {
    const uint32_t g = wave + 4u * k;
    owns[k] = g < uint32_t(G);
    const size_t at = ((size_t(z) * p.kv_heads + h) * G + (owns[k] ? g : 0u)) * 16u + row;
    if constexpr (I8) {
      const int8_t *codes = reinterpret_cast<const int8_t *>(queries) + at * D;
#pragma unroll
      for (int j = 0; j < JQ; ++j) q8[k][j] = *reinterpret_cast<const i32x4 *>(codes + 64 * j + 16 * kq);
      qsum[k] = qsums[at];
    } else {
#pragma unroll
      for (int j = 0; j < JD; ++j) q[k][j] = *reinterpret_cast<const f16x8 *>(queries + at * D + 32 * j + 8 * kq);
      qsum[k] = -(qsums[at] * kCodeOffset);
    }
  }
  const uint32_t ancestors = row < seq.rows ? tree[seq.first_row + row].ancestors : 0u;

  float m[kTiles], l[kTiles];
  f32x4 o[kTiles][DT + 1];
#pragma unroll
  for (int k = 0; k < kTiles; ++k) {
    m[k] = -INFINITY;
    l[k] = 0.f;
#pragma unroll
    for (int dt = 0; dt <= DT; ++dt) o[k][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // A step's loads of this thread: kKeyVectors 16-byte vectors of keys, as many of values, a scale.
  uint4 keyLoad[kKeyVectors], valueLoad[kValueVectors];
  uint32_t scaleLoad = 0;
  // The page table is read one page ahead of the page loop, so that a step's loads never wait
  // for a table entry first (all of this is wave-uniform).
  const uint64_t *entries = page_table + seq.table_first;
  const uint32_t lastPage = total ? (total - 1u) / ATTENTION_PAGE_TOKENS : 0u;
  uint32_t heldPage = min(first / ATTENTION_PAGE_TOKENS, lastPage);
  uint64_t heldEntry = entries[heldPage], nextEntry = entries[min(heldPage + 1u, lastPage)];
  auto load = [&](uint32_t step) {
    const uint32_t token0 = first + step * kStep;
    if (token0 / ATTENTION_PAGE_TOKENS != heldPage) {
      heldPage = token0 / ATTENTION_PAGE_TOKENS;
      heldEntry = nextEntry;
      nextEntry = entries[min(heldPage + 1u, lastPage)];
    }
    uint8_t *page = pool + heldEntry * p.page_bytes;
    const uint32_t inPage = token0 % ATTENTION_PAGE_TOKENS;
    const uint4 *keys = reinterpret_cast<const uint4 *>(page + attention_key_index(h, inPage, 0, D));
    const uint4 *values = reinterpret_cast<const uint4 *>(page + attention_page_values_offset(p.kv_heads, D) +
                                                          attention_value_index(h, inPage, 0, D));
#pragma unroll
    for (int n = 0; n < kKeyVectors; ++n) keyLoad[n] = load_stream(keys + tid + 256u * n);
#pragma unroll
    for (int n = 0; n < kValueVectors; ++n) valueLoad[n] = load_stream(values + tid + 256u * n);
    if (tid < 2 * kStep) {
      const uint16_t *scales = reinterpret_cast<const uint16_t *>(
          page + (tid < kStep ? attention_page_key_scales_offset(p.kv_heads, D) : attention_page_value_scales_offset(p.kv_heads, D)));
      scaleLoad = scales[attention_scale_index(h, inPage + (tid & (kStep - 1)))];
    }
  };
  auto stage = [&](uint32_t buffer) {
#pragma unroll
    for (int n = 0; n < kKeyVectors; ++n) {
      const uint32_t v = tid + 256u * n, token = v / (D / 16), dq = v % (D / 16);
      if constexpr (I8) {
        *reinterpret_cast<uint4 *>(reinterpret_cast<int8_t *>(&ldsK[buffer][token][0]) + 16 * dq) = keyLoad[n];
      } else {
        const uint4 x = make_uint4(keyLoad[n].x ^ 0x80808080u, keyLoad[n].y ^ 0x80808080u, keyLoad[n].z ^ 0x80808080u,
                                   keyLoad[n].w ^ 0x80808080u);
        const uint2 a = bytes_to_f16(x.x), b = bytes_to_f16(x.y), c = bytes_to_f16(x.z), d = bytes_to_f16(x.w);
        uint4 *out = reinterpret_cast<uint4 *>(&ldsK[buffer][token][16 * dq]);
        out[0] = make_uint4(a.x, a.y, b.x, b.y);
        out[1] = make_uint4(c.x, c.y, d.x, d.y);
      }
    }
#pragma unroll
    for (int n = 0; n < kValueVectors; ++n) {
      // 16 tokens (tile tt of the step) of dimension d: token 4 kq' + i of the tile is operand
      // element 4 (tt % 2) + i of lane quarter kq' in token pair-block tt / 2.
      const uint32_t v = tid + 256u * n, d = v / 4u, tt = v % 4u;
      const uint32_t words[4] = {valueLoad[n].x ^ 0x80808080u, valueLoad[n].y ^ 0x80808080u, valueLoad[n].z ^ 0x80808080u,
                                 valueLoad[n].w ^ 0x80808080u};
#pragma unroll
      for (uint32_t quarter = 0; quarter < 4; ++quarter)
        *reinterpret_cast<uint2 *>(&ldsV[buffer][d][((tt >> 1) * 4u + quarter) * 8u + 4u * (tt & 1u)]) = bytes_to_f16(words[quarter]);
    }
    // Key scales carry the softmax scale (log2 domain), value scales the 2^10 of P.
    if (tid < 2 * kStep) (tid < kStep ? ldsKS[buffer] : ldsVS[buffer])[tid & (kStep - 1)] = half_bits_to_float(scaleLoad) * (tid < kStep ? scale2 : kPScale);
  };

  if (steps) {
    load(0);
    stage(0);
  }
  __syncthreads();
  const f16x8 ones = {_Float16(1.f), _Float16(1.f), _Float16(1.f), _Float16(1.f), _Float16(1.f), _Float16(1.f), _Float16(1.f), _Float16(1.f)};
  // One 64-token step. Masked steps (those that reach the block's own rows or the end of the
  // sequence) test every score's visibility; the steps before them, all of the history, do not.
  auto compute = [&](uint32_t buffer, uint32_t token0, auto maskedTag) {
    constexpr bool kMasked = decltype(maskedTag)::value;
    // Scores, transposed: tile tt holds tokens 16 tt + 4 kq + i of the step for fused row `row`.
    // The accumulator starts at -1152 sum(q), which takes the code offset out of the product.
    f32x4 s[kTiles][4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      if constexpr (I8) {
        // the keys' bytes against the queries' codes, exact in int32; the row's scale follows with the key's
        i32x4 key[JQ];
        const int8_t *bytes = reinterpret_cast<const int8_t *>(&ldsK[buffer][16 * tt + row][0]);
#pragma unroll
        for (int j = 0; j < JQ; ++j) key[j] = *reinterpret_cast<const i32x4 *>(bytes + 64 * j + 16 * kq);
#pragma unroll
        for (int k = 0; k < kTiles; ++k) {
          i32x4 acc = {0, 0, 0, 0};
#pragma unroll
          for (int j = 0; j < JQ; ++j) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(key[j], q8[k][j], acc, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) s[k][tt][i] = float(acc[i]) * qsum[k];
        }
      } else {
        f16x8 key[JD];
#pragma unroll
        for (int j = 0; j < JD; ++j) key[j] = *reinterpret_cast<const f16x8 *>(&ldsK[buffer][16 * tt + row][32 * j + 8 * kq]);
#pragma unroll
        for (int k = 0; k < kTiles; ++k) {
          f32x4 acc = {qsum[k], qsum[k], qsum[k], qsum[k]};
#pragma unroll
          for (int j = 0; j < JD; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(key[j], q[k][j], acc, 0, 0, 0);
          s[k][tt] = acc;
        }
      }
    }
    f32x4 keyScale[4], valueScale[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      keyScale[tt] = *reinterpret_cast<const f32x4 *>(&ldsKS[buffer][16 * tt + 4 * kq]);
      valueScale[tt] = *reinterpret_cast<const f32x4 *>(&ldsVS[buffer][16 * tt + 4 * kq]);
    }
    f16x8 pOperand[kTiles][2];
#pragma unroll
    for (int k = 0; k < kTiles; ++k) {
      float stepMax = -INFINITY;
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float score = s[k][tt][i] * keyScale[tt][i];
          if constexpr (kMasked) {
            const uint32_t token = token0 + 16u * tt + 4u * kq + i;
            const bool visible = token < seq.committed || (token < total && ((ancestors >> (token - seq.committed)) & 1u));
            score = visible ? score : -INFINITY;
          }
          s[k][tt][i] = score;
          stepMax = fmaxf(stepMax, score);
        }
      stepMax = fmaxf(stepMax, __shfl_xor(stepMax, 16, 64));
      stepMax = fmaxf(stepMax, __shfl_xor(stepMax, 32, 64));
      const float newMax = fmaxf(m[k], stepMax), safeMax = newMax == -INFINITY ? 0.f : newMax;
      const float alpha = __builtin_amdgcn_exp2f(m[k] - safeMax);
      m[k] = newMax;
      float sum = 0.f;
      float folded[16];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float pr = __builtin_amdgcn_exp2f(s[k][tt][i] - safeMax);
          sum += pr;
          const float f = pr * valueScale[tt][i];
          // A slot past the sequence's end may hold any scale: its weight is zero whatever it is.
          folded[4 * tt + i] = kMasked ? (pr > 0.f ? f : 0.f) : f;
        }
      l[k] = l[k] * alpha + sum;
      // rescale the running output only when some row's maximum grew (paged_attention_tile.h:450-458)
      if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
        for (int dt = 0; dt <= DT; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[k][dt][i] *= alpha;
      }
#pragma unroll
      for (int pair = 0; pair < 2; ++pair)
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          typedef __attribute__((ext_vector_type(2))) float f32x2;
          typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
          const f16x2 two = __builtin_convertvector(f32x2{folded[8 * pair + e], folded[8 * pair + e + 1]}, f16x2);
          pOperand[k][pair][e] = two[0];
          pOperand[k][pair][e + 1] = two[1];
        }
    }
    // Outputs, transposed: o[dt] holds dimensions 16 dt + 4 kq + i of fused row `row`.
#pragma unroll
    for (int pair = 0; pair < 2; ++pair) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const f16x8 value = *reinterpret_cast<const f16x8 *>(&ldsV[buffer][16 * dt + row][(pair * 4 + kq) * 8]);
#pragma unroll
        for (int k = 0; k < kTiles; ++k) o[k][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(value, pOperand[k][pair], o[k][dt], 0, 0, 0);
      }
#pragma unroll
      for (int k = 0; k < kTiles; ++k) o[k][DT] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pOperand[k][pair], o[k][DT], 0, 0, 0);
    }
  };
  // Steps wholly inside the committed history come first, in a loop of their own.
  const uint32_t plain = first < seq.committed ? min(steps, (seq.committed - first) / kStep) : 0u;
  uint32_t step = 0;
  // A SIMD holds one wave of each of a compute unit's two workgroups and issues the older one's instructions first, so
  // the workgroup placed second runs every step behind the first and then finishes alone on an idle unit. The waves
  // take turns instead: a wave's priority is up on the steps whose parity is its wave slot's.
  const uint32_t slot = __builtin_amdgcn_s_getreg((3 << 11) | 4) & 1u;   // HW_ID's wave slot, bit 0
  auto takeTurn = [&](uint32_t s) {
    if ((s + slot) & 1u) __builtin_amdgcn_s_setprio(2);
    else __builtin_amdgcn_s_setprio(0);
  };
  for (; step < plain; ++step) {
    takeTurn(step);
    const uint32_t buffer = step & 1u;
    if (step + 1 < steps) load(step + 1);
    compute(buffer, first + step * kStep, std::false_type{});
    if (step + 1 < steps) stage(buffer ^ 1u);
    __syncthreads();
  }
  for (; step < steps; ++step) {
    takeTurn(step);
    const uint32_t buffer = step & 1u;
    if (step + 1 < steps) load(step + 1);
    compute(buffer, first + step * kStep, std::true_type{});
    if (step + 1 < steps) stage(buffer ^ 1u);
    __syncthreads();
  }

  // The split's partials: the code offset leaves with the row's sum of P, the 2^10 with a scale. The
  // outputs leave divided by the row's sum, a weighted mean of value rows whatever the split's
  // length, as fp16: a lane's 4 DT values are contiguous (position 4 DT kq + 4 dt + i of the row
  // holds dimension 16 dt + 4 kq + i), so a row's 2 D bytes go out as whole 16-byte stores.
#pragma unroll
  for (int k = 0; k < kTiles; ++k) {
    if (!owns[k]) continue;
    const uint32_t g = wave + 4u * k;
    float sum = l[k];
    sum += lane_xor<16>(sum);
    sum += lane_xor<32>(sum);
    const size_t fused = ((size_t(z) * p.kv_heads + h) * p.splits + split) * (16u * G) + 16u * g + row;
    const float rowSum = o[k][DT][0] * kCodeOffset;
    const float norm = sum > 0.f ? 1.0f / (sum * kPScale) : 0.f;
    if constexpr (Whole) {
      // dimensions 16 dt + 4 kq .. + 3 of query head h G + g, four to a store
      if (row >= seq.rows) continue;
      const uint32_t head = h * uint32_t(G) + g;
      const size_t packedRow = size_t(seq.first_row) + row;
      uint2 *mine = reinterpret_cast<uint2 *>(out + packedRow * (p.q_heads * D) + head * D);
      const uint2 *gates = reinterpret_cast<const uint2 *>(packed + packedRow * p.qkv_stride + head * 2u * D + D);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        uint32_t bits[4];
        const uint2 gate = p.gated ? gates[4 * dt + kq] : make_uint2(0u, 0u);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          bits[i] = float_to_bf16_bits((o[k][dt][i] - rowSum) * norm);
          if (p.gated) {
            const float x = bf16_bits_to_float(((i < 2 ? gate.x : gate.y) >> (16 * (i & 1))) & 0xFFFFu);
            bits[i] = float_to_bf16_bits(bf16_bits_to_float(bits[i]) * (1.0f / (1.0f + __builtin_amdgcn_exp2f(-kLog2e * x))));
          }
        }
        mine[4 * dt + kq] = make_uint2(bits[0] | (bits[1] << 16), bits[2] | (bits[3] << 16));
      }
      continue;
    }
    uint4 *mine = reinterpret_cast<uint4 *>(partialO + fused * D + 4u * DT * kq);
#pragma unroll
    for (int dt = 0; dt < DT; dt += 2) {
      f16x8 out;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        out[i] = _Float16((o[k][dt][i] - rowSum) * norm);
        out[4 + i] = _Float16((o[k][dt + 1][i] - rowSum) * norm);
      }
      mine[dt / 2] = __builtin_bit_cast(uint4, out);
    }
    if (kq == 0) {
      partialML[2 * fused] = m[k];
      partialML[2 * fused + 1] = sum;
    }
  }
}
template <int D, int G, bool I8, bool Chunk = false>
__global__ __launch_bounds__(256, 2) void attention_q8_split(const _Float16 *__restrict__ queries, const float *__restrict__ qsums,
                                                          const AttentionTreeRow *__restrict__ tree,
                                                          const uint64_t *__restrict__ page_table, uint8_t *__restrict__ pool,
                                                          _Float16 *__restrict__ partialO, float *__restrict__ partialML,
                                                          AttentionParams p) {
  attention_split<D, G, I8, false, Chunk>(queries, qsums, tree, page_table, pool, partialO, partialML, nullptr, nullptr, p, blockIdx.x, blockIdx.y,
                                   blockIdx.z);
}
// attention_q8_whole: grid (kv_heads * blocks), 256 threads. A prompt chunk's blocks of sixteen rows, each over its whole
// history in one workgroup: no partials, no merge, and the fixed cost of a split (its queries, the first step's latency,
// the partials, about 18 us) once a block. Neighbouring workgroups take the KV heads in turn, so that with eight heads a
// die (workgroup b runs on die b % 8) keeps one head's keys and values in its L2; the longest blocks start first.
template <int D, int G>
__global__ __launch_bounds__(256, 2) void attention_q8_whole(const _Float16 *__restrict__ queries, const float *__restrict__ qsums,
                                                             const AttentionTreeRow *__restrict__ tree,
                                                             const uint64_t *__restrict__ page_table, uint8_t *__restrict__ pool,
                                                             uint16_t *__restrict__ out, const uint16_t *__restrict__ packed,
                                                             AttentionParams p) {
  const uint32_t blocks = gridDim.x / p.kv_heads;
  attention_split<D, G, false, true, true>(queries, qsums, tree, page_table, pool, nullptr, nullptr, out, packed, p, blockIdx.x % p.kv_heads, 0u,
                                     blocks - 1u - blockIdx.x / p.kv_heads);
}
SP_REGISTER_KERNEL("attention_q8_whole_d128_g8", (&attention_q8_whole<128, 8>));
SP_REGISTER_KERNEL("attention_q8_whole_d128_g4", (&attention_q8_whole<128, 4>));
SP_REGISTER_KERNEL("attention_q8_whole_d64_g2", (&attention_q8_whole<64, 2>));
SP_REGISTER_KERNEL("attention_q8_split_d128_g8", &attention_q8_split<128, 8, false>);
SP_REGISTER_KERNEL("attention_q8_split_d128_g4", &attention_q8_split<128, 4, false>);
SP_REGISTER_KERNEL("attention_q8_split_d64_g2", &attention_q8_split<64, 2, false>);
SP_REGISTER_KERNEL("attention_q8_split_chunk_d128_g8", (&attention_q8_split<128, 8, false, true>));
SP_REGISTER_KERNEL("attention_q8_split_chunk_d128_g4", (&attention_q8_split<128, 4, false, true>));
SP_REGISTER_KERNEL("attention_q8_split_chunk_d64_g2", (&attention_q8_split<64, 2, false, true>));
SP_REGISTER_KERNEL("attention_q8q_split_d128_g8", &attention_q8_split<128, 8, true>);
SP_REGISTER_KERNEL("attention_q8q_split_d128_g4", &attention_q8_split<128, 4, true>);
SP_REGISTER_KERNEL("attention_q8q_split_d64_g2", &attention_q8_split<64, 2, true>);

// ---------------------------------------------------------------------------------------------
// attention_q8_few: grid (parts * kv_heads, splits, sequences), 64 threads: the same partials, bit for bit, for blocks of at
// most 16 T parts / G rows, whose (row, head) pairs fill T tiles of sixteen a part where attention_q8_split always computes G
// tiles. The parts of a head read its keys and values each for itself, on one die, whose L2 answers all but the first.
//
// A wave walks its split alone: no staging, no barrier. Keys and values go from the cache's pages straight into registers in
// whole 16-byte loads, and lane-row swaps put them in operand order: of a token's key codes lane quarter a loads chunk a with
// its bits exchanged, and one v_permlane16_swap of the chunk's halves leaves unit 4 j + a of eight codes in quarter a; of a
// dimension's 64 values quarter a loads tokens 16 a .. + 15, and a 4 x 4 transpose (two v_permlane32_swap, two
// v_permlane16_swap) leaves tokens 16 j + 4 a .. + 3. Loads run `Ahead` steps ahead through a buffer resource of their page,
// which past the split's last step is empty (zeros, no traffic), so nothing branches around them.
//
// Bound by memory latency at two waves a compute unit: one row of 64 / 8 heads behind 100000 tokens takes 48 us (4.3 TB/s of
// keys and values, a copy 5.2) against 77 in attention_q8_split, which computes 128 pairs for its eight.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ void swap_rows16(uint32_t &a, uint32_t &b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ void swap_rows32(uint32_t &a, uint32_t &b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
template <int D, int G, int T, int Ahead>
__global__ __launch_bounds__(64, 1) void attention_q8_few(const _Float16 *__restrict__ queries, const float *__restrict__ qsums,
                                                                      const AttentionTreeRow *__restrict__ tree,
                                                                      const uint64_t *__restrict__ page_table, uint8_t *__restrict__ pool,
                                                                      _Float16 *__restrict__ partialO, float *__restrict__ partialML,
                                                                      AttentionParams p) {
  constexpr uint32_t kStep = ATTENTION_STEP_TOKENS;
  constexpr int JD = D / 32, DT = D / 16, KL = D / 64;
  __shared__ __align__(16) float scales[2][kStep];
  const uint32_t lane = threadIdx.x, column = lane & 15u, kq = lane >> 4, h = blockIdx.x % p.kv_heads, part = blockIdx.x / p.kv_heads, split = blockIdx.y, z = blockIdx.z;
  const AttentionSequence seq = p.sequence[z];
  const uint32_t total = seq.committed + seq.rows, span = uint32_t(seq.steps_per_split) * kStep;
  const uint32_t first = min(total, split * span), last = min(total, (split + 1) * span);
  const uint32_t steps = first < last ? (last - first + kStep - 1) / kStep : 0;
  const float scale2 = kLog2e / sqrtf(float(D));

  // Column c of all parts' tiles is row c % rowsHeld of head c / rowsHeld (rowsHeld a power of two).
  const uint32_t rowsShift = uint32_t(__builtin_ctz(gridDim.x / p.kv_heads * (16u * T) / G));
  auto headOf = [&](uint32_t k) { return (16u * (part * T + k) + column) >> rowsShift; };
  const uint32_t row = column & ((1u << rowsShift) - 1u);
  f16x8 q[T][JD];
  float qsum[T];
  uint32_t ancestors[T];
#pragma unroll
  for (int k = 0; k < T; ++k) {
    const size_t at = ((size_t(z) * p.kv_heads + h) * G + headOf(k)) * 16u + row;
#pragma unroll
    for (int j = 0; j < JD; ++j) q[k][j] = *reinterpret_cast<const f16x8 *>(queries + at * D + 32 * j + 8 * kq);
    qsum[k] = -(qsums[at] * kCodeOffset);
    ancestors[k] = row < seq.rows ? tree[seq.first_row + row].ancestors : 0u;
  }
  float m[T], l[T];
  f32x4 o[T][DT + 1];
#pragma unroll
  for (int k = 0; k < T; ++k) {
    m[k] = -INFINITY;
    l[k] = 0.f;
#pragma unroll
    for (int dt = 0; dt <= DT; ++dt) o[k][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  struct Raw {
    uint4 key[4][KL], value[DT];
    uint32_t keyScale, valueScale;   // of token `lane`
  };
  const uint64_t *entries = page_table + seq.table_first;
  const uint32_t lastPage = total ? (total - 1u) / ATTENTION_PAGE_TOKENS : 0u;
  uint32_t heldPage = min(first / ATTENTION_PAGE_TOKENS, lastPage);
  uint64_t heldEntry = entries[heldPage], nextEntry = entries[min(heldPage + 1u, lastPage)];   // (read one page ahead)
  struct Page {
    Resource bytes;
    uint32_t inPage;
  };
  auto pageOf = [&](uint32_t step) __attribute__((always_inline)) {
    const uint32_t token0 = first + step * kStep;
    if (step < steps && token0 / ATTENTION_PAGE_TOKENS != heldPage) {
      heldPage = token0 / ATTENTION_PAGE_TOKENS;
      heldEntry = nextEntry;
      nextEntry = entries[min(heldPage + 1u, lastPage)];
    }
    return Page{make_resource(pool + heldEntry * p.page_bytes, step < steps ? uint32_t(attention_page_bytes(p.kv_heads, D)) : 0u), token0 % ATTENTION_PAGE_TOKENS};
  };
  const uint32_t keyLane = column * D + 16u * (((kq & 1u) << 1) | (kq >> 1)), valueLane = column * kStep + 16u * kq;
  auto loadKeys = [&](Raw &raw, const Page &page) __attribute__((always_inline)) {
    const uint32_t at = uint32_t(attention_key_index(h, page.inPage, 0, D)) + keyLane;
#pragma unroll
    for (uint32_t tt = 0; tt < 4; ++tt)
#pragma unroll
      for (uint32_t n = 0; n < KL; ++n) raw.key[tt][n] = load128<0>(page.bytes, at + tt * (16u * D) + 64u * n);
    raw.keyScale = __builtin_amdgcn_raw_buffer_load_b16(
        page.bytes, int(uint32_t(attention_page_key_scales_offset(p.kv_heads, D)) + 2u * (uint32_t(attention_scale_index(h, page.inPage)) + lane)), 0, 0);
    raw.valueScale = __builtin_amdgcn_raw_buffer_load_b16(
        page.bytes, int(uint32_t(attention_page_value_scales_offset(p.kv_heads, D)) + 2u * (uint32_t(attention_scale_index(h, page.inPage)) + lane)), 0, 0);
  };
  auto loadValues = [&](Raw &raw, const Page &page) __attribute__((always_inline)) {
    const uint32_t at = uint32_t(attention_page_values_offset(p.kv_heads, D)) + uint32_t(attention_value_index(h, page.inPage, 0, D)) + valueLane;
#pragma unroll
    for (uint32_t dt = 0; dt < uint32_t(DT); ++dt) raw.value[dt] = load128<kStreamOnce>(page.bytes, at + dt * (16u * kStep));
  };
  const f16x8 ones = {_Float16(1.f), _Float16(1.f), _Float16(1.f), _Float16(1.f), _Float16(1.f), _Float16(1.f), _Float16(1.f), _Float16(1.f)};
  auto operand = [](uint32_t a, uint32_t b) __attribute__((always_inline)) {   // two words of codes as 1152 + code
    const uint2 x = bytes_to_f16(a ^ 0x80808080u), y = bytes_to_f16(b ^ 0x80808080u);
    return __builtin_bit_cast(f16x8, make_uint4(x.x, x.y, y.x, y.y));
  };

  // One step, its arithmetic attention_split's (see there); `raw` then takes the step `Ahead` after it.
  auto run = [&](uint32_t step, Raw &raw, auto maskedTag) __attribute__((always_inline)) {
    constexpr bool kMasked = decltype(maskedTag)::value;
    const Page next = pageOf(step + Ahead);
    wave_lds_fence();
    scales[0][lane] = half_bits_to_float(raw.keyScale) * scale2;
    scales[1][lane] = half_bits_to_float(raw.valueScale) * kPScale;
    wave_lds_fence();
    f32x4 s[T][4];
#pragma unroll
    for (uint32_t tt = 0; tt < 4; ++tt) {
      f16x8 key[JD];
#pragma unroll
      for (uint32_t n = 0; n < KL; ++n) {
        uint4 x = raw.key[tt][n];
        swap_rows16(x.x, x.z);
        swap_rows16(x.y, x.w);
        key[2 * n] = operand(x.x, x.y);
        key[2 * n + 1] = operand(x.z, x.w);
      }
#pragma unroll
      for (int k = 0; k < T; ++k) {
        f32x4 acc = {qsum[k], qsum[k], qsum[k], qsum[k]};
#pragma unroll
        for (int j = 0; j < JD; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(key[j], q[k][j], acc, 0, 0, 0);
        s[k][tt] = acc;
      }
    }
    loadKeys(raw, next);
    f32x4 keyScale[4], valueScale[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      keyScale[tt] = *reinterpret_cast<const f32x4 *>(&scales[0][16 * tt + 4 * kq]);
      valueScale[tt] = *reinterpret_cast<const f32x4 *>(&scales[1][16 * tt + 4 * kq]);
    }
    f16x8 pOperand[T][2];
#pragma unroll
    for (int k = 0; k < T; ++k) {
      float stepMax = -INFINITY;
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float score = s[k][tt][i] * keyScale[tt][i];
          if constexpr (kMasked) {
            const uint32_t token = first + step * kStep + 16u * tt + 4u * kq + i;
            const bool visible = token < seq.committed || (token < total && ((ancestors[k] >> (token - seq.committed)) & 1u));
            score = visible ? score : -INFINITY;
          }
          s[k][tt][i] = score;
          stepMax = fmaxf(stepMax, score);
        }
      stepMax = fmaxf(stepMax, __shfl_xor(stepMax, 16, 64));
      stepMax = fmaxf(stepMax, __shfl_xor(stepMax, 32, 64));
      const float newMax = fmaxf(m[k], stepMax), safeMax = newMax == -INFINITY ? 0.f : newMax;
      const float alpha = __builtin_amdgcn_exp2f(m[k] - safeMax);
      m[k] = newMax;
      float sum = 0.f, folded[16];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float pr = __builtin_amdgcn_exp2f(s[k][tt][i] - safeMax);
          sum += pr;
          const float f = pr * valueScale[tt][i];
          folded[4 * tt + i] = kMasked ? (pr > 0.f ? f : 0.f) : f;
        }
      l[k] = l[k] * alpha + sum;
      if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
        for (int dt = 0; dt <= DT; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[k][dt][i] *= alpha;
      }
#pragma unroll
      for (int pair = 0; pair < 2; ++pair)
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          typedef __attribute__((ext_vector_type(2))) float f32x2;
          typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
          const f16x2 two = __builtin_convertvector(f32x2{folded[8 * pair + e], folded[8 * pair + e + 1]}, f16x2);
          pOperand[k][pair][e] = two[0];
          pOperand[k][pair][e + 1] = two[1];
        }
    }
#pragma unroll
    for (uint32_t dt = 0; dt < uint32_t(DT); ++dt) {
      uint4 x = raw.value[dt];
      swap_rows32(x.x, x.z);
      swap_rows32(x.y, x.w);
      swap_rows16(x.x, x.y);
      swap_rows16(x.z, x.w);
      const f16x8 value[2] = {operand(x.x, x.y), operand(x.z, x.w)};
#pragma unroll
      for (int k = 0; k < T; ++k)
#pragma unroll
        for (int pair = 0; pair < 2; ++pair) o[k][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(value[pair], pOperand[k][pair], o[k][dt], 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < T; ++k)
#pragma unroll
      for (int pair = 0; pair < 2; ++pair) o[k][DT] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pOperand[k][pair], o[k][DT], 0, 0, 0);
    loadValues(raw, next);
  };
  Raw raw[Ahead];
#pragma unroll
  for (uint32_t a = 0; a < uint32_t(Ahead); ++a) {
    const Page page = pageOf(a);
    loadKeys(raw[a], page);
    loadValues(raw[a], page);
    __builtin_amdgcn_sched_barrier(0);   // (in the order the loop waits for them)
  }
  // Steps wholly inside the committed history, then those that reach the block's own rows or the sequence's end.
  const uint32_t plain = first < seq.committed ? min(steps, (seq.committed - first) / kStep) : 0u;
  for (uint32_t step = 0; step < steps; step += Ahead) {
#pragma unroll
    for (uint32_t a = 0; a < uint32_t(Ahead); ++a) {
      if (step + a < plain) run(step + a, raw[a], std::false_type{});
      else if (step + a < steps) run(step + a, raw[a], std::true_type{});
    }
  }

  // The partials, as attention_split leaves them.
#pragma unroll
  for (int k = 0; k < T; ++k) {
    const uint32_t g = headOf(k);
    float sum = l[k];
    sum += lane_xor<16>(sum);
    sum += lane_xor<32>(sum);
    if (row >= seq.rows) continue;
    const size_t fused = ((size_t(z) * p.kv_heads + h) * p.splits + split) * (16u * G) + 16u * g + row;
    const float rowSum = o[k][DT][0] * kCodeOffset, norm = sum > 0.f ? 1.0f / (sum * kPScale) : 0.f;
    uint4 *mine = reinterpret_cast<uint4 *>(partialO + fused * D + 4u * DT * kq);
#pragma unroll
    for (int dt = 0; dt < DT; dt += 2) {
      f16x8 out;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        out[i] = _Float16((o[k][dt][i] - rowSum) * norm);
        out[4 + i] = _Float16((o[k][dt + 1][i] - rowSum) * norm);
      }
      mine[dt / 2] = __builtin_bit_cast(uint4, out);
    }
    if (kq == 0) {
      partialML[2 * fused] = m[k];
      partialML[2 * fused + 1] = sum;
    }
  }
}
SP_REGISTER_KERNEL("attention_q8_few_d128_g8_t1", (&attention_q8_few<128, 8, 1, 2>));
SP_REGISTER_KERNEL("attention_q8_few_d128_g8_t2", (&attention_q8_few<128, 8, 2, 2>));
SP_REGISTER_KERNEL("attention_q8_few_d128_g4_t1", (&attention_q8_few<128, 4, 1, 2>));
SP_REGISTER_KERNEL("attention_q8_few_d128_g4_t2", (&attention_q8_few<128, 4, 2, 2>));
SP_REGISTER_KERNEL("attention_q8_few_d64_g2_t1", (&attention_q8_few<64, 2, 1, 2>));

// ---------------------------------------------------------------------------------------------
// attention_reduce: grid (q_heads, 16, sequences), 256 threads. Merges the splits of one (head,
// row) in a fixed order (paged_attention_tile.h:499-535) and writes bf16 [packed row][q_heads * D].
// Thread (part, quad) sums splits part, part + P, ... of the row's positions 4 quad .. 4 quad + 3
// (four dimensions in a row, in the order the split kernel leaves them), all its loads in flight
// together; the P parts are then added in part order. A split weighs exp2(its maximum - the
// largest) times its sum: its outputs arrive divided by that sum.
// ---------------------------------------------------------------------------------------------
// The _t variant also writes the rows as the activation table (abi/Gguf.h) of the projection that
// follows, as gguf_prepare_table would from `out`; p.table_tiles is the table's row tiles. Rows of
// a tile past the packed rows keep what the table held.
template <int D, bool Table, bool Chunk = false>
__global__ __launch_bounds__(256) void attention_reduce(const _Float16 *__restrict__ partialO, const float *__restrict__ partialML,
                                                        uint16_t *__restrict__ out, uint8_t *__restrict__ table,
                                                        const uint16_t *__restrict__ qkv, AttentionParams p) {
  constexpr uint32_t kQuads = D / 4, kParts = 256 / kQuads;
  __shared__ float weights[ATTENTION_MAXIMUM_SPLITS];
  __shared__ float scratch[4];
  __shared__ __align__(16) float4 sums[kParts][kQuads];
  __shared__ uint16_t staged[D];
  const uint32_t tid = threadIdx.x, head = blockIdx.x, row = blockIdx.y, z = blockIdx.z;
  const AttentionSequence seq = block_sequence<Chunk>(p, z);
  if (row >= seq.rows) return;
  const uint32_t group = p.q_heads / p.kv_heads, h = head / group, g = head % group, fusedRows = 16u * group;
  const size_t base = (size_t(z) * p.kv_heads + h) * p.splits;
  auto fusedOf = [&](uint32_t s) { return (base + s) * fusedRows + 16u * g + row; };

  // Split tid's maximum and sum; the block's maximum; the split's weight and its share of the denominator.
  float ms = -INFINITY, ls = 0.f;
  if (tid < p.splits) {
    const float2 ml = *reinterpret_cast<const float2 *>(partialML + 2 * fusedOf(tid));
    ms = ml.x;
    ls = ml.y;
  }
  const float maximum = block_max<256>(ms, scratch, tid);
  const float weight = ms == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms - maximum);
  if (tid < ATTENTION_MAXIMUM_SPLITS) weights[tid] = weight * ls;
  const float denominator = block_sum<256>(weight * ls, scratch, tid);  // block_sum's barriers publish the weights too

  const uint32_t part = tid / kQuads, quad = tid % kQuads;
  float4 total = make_float4(0.f, 0.f, 0.f, 0.f);
  typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
  for (uint32_t s0 = part; s0 < p.splits; s0 += 4u * kParts) {
    uint2 held[4];
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) {
      const uint32_t s = s0 + i * kParts;
      held[i] = s < p.splits ? reinterpret_cast<const uint2 *>(partialO + fusedOf(s) * D)[quad] : make_uint2(0u, 0u);
    }
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) {
      const uint32_t s = s0 + i * kParts;
      const float w = s < p.splits ? weights[s] : 0.f;
      if (w != 0.f) {  // a split without a visible token may hold anything
        const f16x4 x = __builtin_bit_cast(f16x4, held[i]);
        total.x += w * float(x[0]);
        total.y += w * float(x[1]);
        total.z += w * float(x[2]);
        total.w += w * float(x[3]);
      }
    }
  }
  // position quad of the row is dimensions 16 (quad % DT) + 4 (quad / DT) ..
  sums[part][4u * (quad % (D / 16u)) + quad / (D / 16u)] = total;
  __syncthreads();
  if (tid < D) {
    const float *flat = reinterpret_cast<const float *>(&sums[0][0]);
    float numerator = 0.f;
#pragma unroll
    for (uint32_t q = 0; q < kParts; ++q) numerator += flat[q * D + tid];
    const float value = denominator > 0.f ? numerator / denominator : 0.f;
    uint32_t bits = float_to_bf16_bits(value);
    if (p.gated) {
      // attention_gate.h:27-31: bf16(value) times the sigmoid of the head's gate in the row's packed projection.
      const float gate = bf16_bits_to_float(qkv[(size_t(seq.first_row) + row) * p.qkv_stride + head * 2u * D + D + tid]);
      bits = float_to_bf16_bits(bf16_bits_to_float(bits) * (1.0f / (1.0f + __builtin_amdgcn_exp2f(-kLog2e * gate))));
    }
    out[(size_t(seq.first_row) + row) * (p.q_heads * D) + head * D + tid] = uint16_t(bits);
    if constexpr (Table) staged[tid] = uint16_t(bits);
  }
  if constexpr (Table) {
    __syncthreads();
    if (tid < D / 4u) {
      // Run q: inputs 4 q .. 4 q + 3 of the packed row (norm_rms_table16 writes the same pieces).
      const uint32_t width = p.q_heads * D, G = width / 32u, q = head * (D / 4u) + tid;
      // Row tile packed / 16 is a tile of its 64-row piece's table, which holds `tiles` row tiles.
      const uint32_t packed = seq.first_row + row, r = packed % 16u;
      const uint32_t piece = packed / 16u / GGUF_PIECE_TILES, tile = packed / 16u % GGUF_PIECE_TILES;
      const uint32_t tiles = min(uint32_t(GGUF_PIECE_TILES), p.table_tiles - piece * GGUF_PIECE_TILES);
      uint8_t *mine = table + piece * gguf_table_bytes(width, GGUF_PIECE_TILES);
      const uint32_t x0 = staged[4 * tid], x1 = staged[4 * tid + 1], x2 = staged[4 * tid + 2], x3 = staged[4 * tid + 3];
      const uint32_t g = q / 8u, half = (q / 4u) % 2u, kq = q % 4u;
      reinterpret_cast<uint2 *>(mine)[((size_t(tile) * G + g) * 64u + kq * 16u + r) * 2u + half] = make_uint2(x0 | (x2 << 16), x1 | (x3 << 16));
      float s = (bf16_bits_to_float(x0) + bf16_bits_to_float(x1)) + (bf16_bits_to_float(x2) + bf16_bits_to_float(x3));
      const float s1 = lane_down<1>(s), s2 = lane_down<2>(s), s3 = lane_down<3>(s);
      s = ((s + s1) + s2) + s3;
      const float other = lane_down<4>(s);
      if (kq == 0) {
        float *sums32 = reinterpret_cast<float *>(mine + gguf_table_sums32_offset(width, tiles));
        float *sums16 = reinterpret_cast<float *>(mine + gguf_table_sums16_offset(width, tiles));
        sums16[(size_t(tile) * 2u * G + 2u * g + half) * 16u + r] = s;
        if (half == 0) sums32[(size_t(tile) * G + g) * 16u + r] = s + other;
      }
    }
  }
}
SP_REGISTER_KERNEL("attention_reduce_d128", &attention_reduce<128, false>);
SP_REGISTER_KERNEL("attention_reduce_d64", &attention_reduce<64, false>);
SP_REGISTER_KERNEL("attention_reduce_chunk_d128", (&attention_reduce<128, false, true>));
SP_REGISTER_KERNEL("attention_reduce_chunk_d64", (&attention_reduce<64, false, true>));
SP_REGISTER_KERNEL("attention_reduce_d128_t", &attention_reduce<128, true>);
SP_REGISTER_KERNEL("attention_reduce_d64_t", &attention_reduce<64, true>);

// ---------------------------------------------------------------------------------------------
// attention_q8_commit: grid (kv_heads, sequences, layers), D threads. retained[z] is the mask of the block
// rows on the accepted path; its k-th set bit (row r) moves from slot committed + r to committed + k.
// ---------------------------------------------------------------------------------------------
template <int D>
__device__ __forceinline__ void commit_path(uint32_t mask, const uint64_t *__restrict__ page_table, uint8_t *__restrict__ pool,
                                            const AttentionCommitParams &p) {
  const uint32_t tid = threadIdx.x, h = blockIdx.x, z = blockIdx.y;
  const AttentionSequence seq = p.sequence[z];
  pool += uint64_t(blockIdx.z) * p.layer_bytes;
  uint32_t depth = 0;
  while (mask) {
    const uint32_t r = uint32_t(__builtin_ctz(mask));
    mask &= mask - 1u;
    if (r != depth && r < seq.rows) {
      const uint32_t from = seq.committed + r, to = seq.committed + depth;
      uint8_t *source = page_of(pool, page_table, seq, p.page_bytes, from / ATTENTION_PAGE_TOKENS);
      uint8_t *target = page_of(pool, page_table, seq, p.page_bytes, to / ATTENTION_PAGE_TOKENS);
      const uint32_t ft = from % ATTENTION_PAGE_TOKENS, tt = to % ATTENTION_PAGE_TOKENS;
      target[attention_key_index(h, tt, tid, D)] = source[attention_key_index(h, ft, tid, D)];
      const uint64_t values = attention_page_values_offset(p.kv_heads, D);
      target[values + attention_value_index(h, tt, tid, D)] = source[values + attention_value_index(h, ft, tid, D)];
      if (tid < 2) {
        const uint64_t scales = tid ? attention_page_value_scales_offset(p.kv_heads, D) : attention_page_key_scales_offset(p.kv_heads, D);
        reinterpret_cast<uint16_t *>(target + scales)[attention_scale_index(h, tt)] =
            reinterpret_cast<const uint16_t *>(source + scales)[attention_scale_index(h, ft)];
      }
    }
    ++depth;
    __syncthreads();
  }
}
template <int D>
__global__ __launch_bounds__(D) void attention_q8_commit(const uint32_t *__restrict__ retained,
                                                         const uint64_t *__restrict__ page_table, uint8_t *__restrict__ pool,
                                                         AttentionCommitParams p) {
  commit_path<D>(retained[blockIdx.y], page_table, pool, p);
}

// attention_q8_accept_commit: decode_sample_argmax_reduce, decode_accept_tree and attention_q8_commit of a step whose
// rows are all greedy, on the commit's grid: every workgroup reduces the shards' partials of its lane's rows (half a
// wavefront a row, 4 KB from L2 at most) and walks the block itself, and the first of a lane writes the results the other
// two kernels leave. Two launches of a few waiting wavefronts less a step:
// 6.8 us for 2.8 + 4.5 + 4.1 at 16 rows of one lane. (With the ends' other launches, a step of 8 layers of 5120 columns
// 1296 -> 1286 us.)
template <int D>
__global__ __launch_bounds__(D) void attention_q8_accept_commit(const float *__restrict__ partial_values, const uint32_t *__restrict__ partial_indices,
                                                                const uint32_t *__restrict__ input_tokens, const AttentionTreeRow *__restrict__ tree,
                                                                uint32_t *__restrict__ tokens, uint32_t *__restrict__ retained,
                                                                uint32_t *__restrict__ accepted_count, uint32_t *__restrict__ retained_rows,
                                                                const uint64_t *__restrict__ page_table, uint8_t *__restrict__ pool,
                                                                AttentionAcceptCommitParams p) {
  static_assert(SAMPLING_SHARDS == 32, "half a wavefront holds a row's shards");
  constexpr uint32_t kTogether = D / SAMPLING_SHARDS;   // rows reduced at a time
  __shared__ uint32_t selections[SAMPLING_MAXIMUM_ROWS];
  const uint32_t tid = threadIdx.x, z = blockIdx.y;
  const uint32_t first = p.commit.sequence[z].first_row, rows = min(uint32_t(p.commit.sequence[z].rows), SAMPLING_MAXIMUM_ROWS);
  const uint32_t row = tid & 63u;   // each wavefront walks the whole block
  const bool live = row < rows;
  const AttentionTreeRow node = live ? tree[first + row] : AttentionTreeRow{0u, 0u, 0u};
  const uint32_t input = live ? input_tokens[first + row] : 0u;
  Best best[SAMPLING_MAXIMUM_ROWS / kTogether];
#pragma unroll
  for (uint32_t i = 0; i < SAMPLING_MAXIMUM_ROWS / kTogether; ++i) {
    const uint32_t r = i * kTogether + tid / SAMPLING_SHARDS, at = (first + min(r, rows - 1u)) * SAMPLING_SHARDS + tid % SAMPLING_SHARDS;
    best[i] = {partial_values[at], partial_indices[at]};
  }
#pragma unroll
  for (uint32_t i = 0; i < SAMPLING_MAXIMUM_ROWS / kTogether; ++i) {
    if (unselectable(best[i].value)) best[i] = {-INFINITY, SAMPLING_NO_TOKEN};
    best[i] = wave_best<SAMPLING_SHARDS>(best[i]);
    if (tid % SAMPLING_SHARDS == 0) selections[i * kTogether + tid / SAMPLING_SHARDS] = best[i].index;
  }
  __syncthreads();
  const uint32_t selection = live ? selections[row] : 0u;
  const Acceptance a = accept_rows(row, live, node, input, selection, p.remaining[z], p.stop_tokens);
  if (tid < 64u && blockIdx.x == 0 && blockIdx.z == 0) {
    // the kept path's selections from the lane's first row on, every row past them its own
    if (live && row >= a.kept) tokens[first + row] = selection;
    if (a.retains) tokens[first + a.depth] = selection;
    if (a.last) {
      retained_rows[z] = node.ancestors;
      retained[z] = a.kept;
      accepted_count[z] = a.accepted;
    }
  }
  // a block that keeps no row (its anchor is not its own ancestor) writes no results: the commit reads those that are there
  const uint64_t keeps = __builtin_amdgcn_ballot_w64(a.last);
  const uint32_t mask = keeps ? uint32_t(__shfl(node.ancestors, int(__builtin_ctzll(keeps)), 64)) : retained_rows[z];
  commit_path<D>(mask, page_table, pool, p.commit);
}
SP_REGISTER_KERNEL("attention_q8_accept_commit_d128", &attention_q8_accept_commit<128>);
SP_REGISTER_KERNEL("attention_q8_accept_commit_d64", &attention_q8_accept_commit<64>);
SP_REGISTER_KERNEL("attention_q8_commit_d128", &attention_q8_commit<128>);
SP_REGISTER_KERNEL("attention_q8_commit_d64", &attention_q8_commit<64>);

} // namespace splash::kernels
