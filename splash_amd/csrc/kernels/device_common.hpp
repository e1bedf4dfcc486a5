// Scalar conversions, MFMA operand types and wavefront reductions shared by the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>
#include "abi/Glue.h"

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

// Data that moves between lanes by DPP row permutations and the swaps of 16- and 32-lane rows, a few cycles each, where the
// LDS crossbar (__shfl) takes a hundred. A lane no shift reaches keeps its own value.
template <int Control> __device__ __forceinline__ uint32_t dpp_move(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(v), static_cast<int>(v), Control, 0xF, 0xF, false));
}
constexpr int kRowShiftRight = 0x110, kRowBroadcast15 = 0x142, kRowBroadcast31 = 0x143;
constexpr int kQuadSwap1 = 0xB1, kQuadSwap2 = 0x4E, kRowMirror = 0x140, kRowHalfMirror = 0x141;
constexpr int kRowRotate4 = 0x124, kRowRotate8 = 0x128, kQuadReverse = 0x1B;
__device__ __forceinline__ uint32_t lane_bits(uint32_t v) { return v; }
__device__ __forceinline__ uint32_t lane_bits(int v) { return static_cast<uint32_t>(v); }
__device__ __forceinline__ uint32_t lane_bits(float v) { return __float_as_uint(v); }
template <class T> __device__ __forceinline__ T from_lane_bits(uint32_t v) { return __builtin_bit_cast(T, v); }
// The value of lane (mine ^ Distance).
template <int Distance, class T> __device__ __forceinline__ T lane_xor(T value) {
  static_assert(sizeof(T) == 4);
  const uint32_t v = lane_bits(value), lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  uint32_t other;
  if constexpr (Distance == 1) other = dpp_move<kQuadSwap1>(v);
  else if constexpr (Distance == 2) other = dpp_move<kQuadSwap2>(v);
  else if constexpr (Distance == 4) other = dpp_move<kQuadReverse>(dpp_move<kRowHalfMirror>(v));
  else if constexpr (Distance == 8) other = dpp_move<kRowRotate8>(v);
  else if constexpr (Distance == 16) {
    const auto rows = __builtin_amdgcn_permlane16_swap(v, v, false, false);   // [0]: every pair's first row twice, [1]: its second
    other = lane & 16u ? rows[0] : rows[1];
  } else {
    static_assert(Distance == 32);
    const auto rows = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    other = lane & 32u ? rows[0] : rows[1];
  }
  return from_lane_bits<T>(other);
}
// The value of the lane `Distance` on, of the same sixteen (past their end: a lane's own).
template <int Distance, class T> __device__ __forceinline__ T lane_down(T value) {
  static_assert(sizeof(T) == 4 && Distance > 0 && Distance < 16);
  return from_lane_bits<T>(dpp_move<0x100 + Distance>(lane_bits(value)));
}
// Lane `from`'s value, in every lane.
template <class T> __device__ __forceinline__ T lane_value_of(T value, int from) {
  return from_lane_bits<T>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(lane_bits(value)), from)));
}

// A butterfly over lanes 32, 16, 8, 4, 2 and 1 apart. (A sum is the same whichever of a pair comes first; behind the third
// step a lane's value is that of every lane 8 apart, so a rotation by 4 fetches what lies 4 away.)
template <class T> __device__ __forceinline__ T wave_sum(T v) {
  static_assert(sizeof(T) == 4);
  const auto add = [](uint32_t a, uint32_t b) { return lane_bits(T(from_lane_bits<T>(a) + from_lane_bits<T>(b))); };
  uint32_t u = lane_bits(v);
  const auto halves = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  u = add(halves[0], halves[1]);
  const auto rows = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  u = add(rows[0], rows[1]);
  u = add(u, dpp_move<kRowRotate8>(u));
  u = add(u, dpp_move<kRowRotate4>(u));
  u = add(u, dpp_move<kQuadSwap2>(u));
  u = add(u, dpp_move<kQuadSwap1>(u));
  return from_lane_bits<T>(u);
}
template <class T> __device__ __forceinline__ T wave_max(T v) {
  const auto larger = [](T mine, T other) { return other > mine ? other : mine; };
  v = larger(v, lane_xor<32>(v));
  v = larger(v, lane_xor<16>(v));
  v = larger(v, lane_xor<8>(v));
  v = larger(v, lane_xor<4>(v));
  v = larger(v, lane_xor<2>(v));
  return larger(v, lane_xor<1>(v));
}

// Maxima by shifts and broadcasts along a wavefront's rows, for reductions that follow one another, each waiting for the last.
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
// In the first sixteen lanes: their value, and those of the lanes 16, 32 and 48 on, added in that order.
__device__ __forceinline__ float quarters_sum(float v) {
  const float second = lane_xor<16>(v), third = lane_xor<32>(v), fourth = lane_xor<32>(second);
  return ((v + second) + third) + fourth;
}
// A wavefront's LDS writes before its later reads (its LDS operations are carried out in order).
__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

// The row's inverse RMS: a workgroup's first 256 threads sum the squares of columns tid, tid + 256, ... in column
// order; a wavefront sums its lanes by butterfly, the four wavefronts' sums are added in order
// (normalization.metal:59-99 and common/rms_inverse.h:15-33, on 64-lane wavefronts). The order is the same whatever the
// workgroup's size is.
__device__ __forceinline__ float rms_inverse(const uint16_t *row, uint32_t width, float *scratch) {
  // (ten reads at a time: a column past the row adds a zero)
  constexpr uint32_t kAhead = 10;
  if (threadIdx.x < 256u) {
    float sum = 0.f;
    for (uint32_t first = threadIdx.x; first < width; first += 256u * kAhead) {
      float v[kAhead];
#pragma unroll
      for (uint32_t j = 0; j < kAhead; ++j) v[j] = bf16_bits_to_float(row[min(first + 256u * j, width - 1u)]);
#pragma unroll
      for (uint32_t j = 0; j < kAhead; ++j) sum += first + 256u * j < width ? v[j] * v[j] : 0.f;
    }
    sum = wave_sum(sum);
    if ((threadIdx.x & 63u) == 0) scratch[threadIdx.x >> 6] = sum;
  }
  __syncthreads();
  const float total = ((scratch[0] + scratch[1]) + scratch[2]) + scratch[3];
  return 1.0f / sqrtf(total / float(width) + SPLASH_RMS_EPSILON);
}

} // namespace splash::kernels
