// Scalar conversions, MFMA operand types and wavefront reductions shared by the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

namespace splash::kernels {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(4))) int i32x4;

constexpr int kWave = 64;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

// A 128-bit load of data read once (weights, KV pages): the non-temporal hint keeps it from
// displacing the activations every wave re-reads from the caches.
__device__ __forceinline__ uint4 load_stream(const uint4 *p) {
  const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ float half_bits_to_float(uint32_t bits) {
  return __half2float(__ushort_as_half(static_cast<unsigned short>(bits)));
}
__device__ __forceinline__ uint32_t float_to_half_bits(float v) { return __half_as_ushort(__float2half_rn(v)); }
__device__ __forceinline__ float bf16_bits_to_float(uint32_t bits) { return __uint_as_float(bits << 16); }
// Round to nearest even; NaN stays NaN (its upper bits, quiet): the machine's own conversion, of all 2^32 values the same
// bits as adding 0x7FFF and the last kept bit.
__device__ __forceinline__ uint32_t float_to_bf16_bits(float v) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(v)); }
__device__ __forceinline__ float round_bf16(float v) { return bf16_bits_to_float(float_to_bf16_bits(v)); }

// x / (1 + 2^(-log2(e) x)), the reference's silu (kernels/common/activation.h:8-16).
__device__ __forceinline__ float silu(float x) { return x / (1.0f + exp2f(-1.4426950408889634f * x)); }

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

template <class T> __device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
template <class T> __device__ __forceinline__ T wave_max(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) { const T other = __shfl_xor(v, o, 64); v = other > v ? other : v; }
  return v;
}

// Maxima that move data between lanes with DPP row permutations and broadcasts, a few cycles each, and never through the
// LDS crossbar: for reductions that follow one another, each waiting for the last. A lane no shift reaches keeps its own
// value, which a maximum does not mind.
template <int Control> __device__ __forceinline__ uint32_t dpp_move(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(v), static_cast<int>(v), Control, 0xF, 0xF, false));
}
constexpr int kRowShiftRight = 0x110, kRowBroadcast15 = 0x142, kRowBroadcast31 = 0x143;
constexpr int kQuadSwap1 = 0xB1, kQuadSwap2 = 0x4E, kRowMirror = 0x140, kRowHalfMirror = 0x141;
template <int Control> __device__ __forceinline__ uint32_t dpp_max(uint32_t v) { return max(v, dpp_move<Control>(v)); }
template <int Control> __device__ __forceinline__ uint64_t dpp_max(uint64_t key) {
  const uint64_t other = (uint64_t{dpp_move<Control>(static_cast<uint32_t>(key >> 32))} << 32) | dpp_move<Control>(static_cast<uint32_t>(key));
  return other > key ? other : key;
}
// The largest of a wavefront, in every lane: after the shifts by 1, 2, 4 and 8 a row's last lane holds the row's largest,
// after the two broadcasts lane 63 the wavefront's.
template <class T> __device__ __forceinline__ T wave_max_dpp(T v) {
  v = dpp_max<kRowShiftRight + 1>(v);
  v = dpp_max<kRowShiftRight + 2>(v);
  v = dpp_max<kRowShiftRight + 4>(v);
  v = dpp_max<kRowShiftRight + 8>(v);
  v = dpp_max<kRowBroadcast15>(v);
  v = dpp_max<kRowBroadcast31>(v);
  const uint32_t low = __builtin_amdgcn_readlane(static_cast<int>(static_cast<uint32_t>(v)), 63);
  if constexpr (sizeof(T) == 4) return low;
  else return (uint64_t{uint32_t(__builtin_amdgcn_readlane(static_cast<int>(static_cast<uint32_t>(v >> 32)), 63))} << 32) | low;
}
// The largest of each row of sixteen lanes, in every lane of the row.
__device__ __forceinline__ uint32_t row_max_dpp(uint32_t v) {
  return dpp_max<kRowMirror>(dpp_max<kRowHalfMirror>(dpp_max<kQuadSwap2>(dpp_max<kQuadSwap1>(v))));
}
// The sum of each row of sixteen lanes, in every lane of the row: the additions of a butterfly over lanes 1, 2, 4 and 8 apart
// (behind the first two steps a quad's lanes hold the same sum, behind the third an octet's, so a mirrored lane holds what
// the lane 4 or 8 away does), without the LDS crossbar's latency a step.
template <int Control> __device__ __forceinline__ float dpp_add(float v) { return v + __uint_as_float(dpp_move<Control>(__float_as_uint(v))); }
__device__ __forceinline__ float row_sum_dpp(float v) {
  return dpp_add<kRowMirror>(dpp_add<kRowHalfMirror>(dpp_add<kQuadSwap2>(dpp_add<kQuadSwap1>(v))));
}
// A wavefront's LDS writes before its later reads (its LDS operations are carried out in order).
__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

} // namespace splash::kernels
