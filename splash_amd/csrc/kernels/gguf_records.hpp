// Weight-image records in registers (abi/Gguf.h): how a wave loads a column tile's super-block and turns it into operands,
// shared by every projection kernel.
#pragma once
#include "kernels/gguf_device.hpp"
#include <utility>

namespace splash::kernels {

// ---------------------------------------------------------------------------------------------
// Records in registers.
// ---------------------------------------------------------------------------------------------
// A wave's cursors into one column tile's record stream: its lane's 16 bytes of each 1024-byte
// part, and its column's scale fields. They advance one record per super-block.
template <uint32_t FMT> struct Cursor {
  const uint4 *mine = nullptr;
  const uint4 *column = nullptr;
  const uint16_t *d = nullptr;   // Q6_K only
  const uint2 *fifth = nullptr;  // Q5_K only
  const uint2 *meta8 = nullptr;  // IQ4_XS only: its column's eight bytes
  static constexpr uint32_t kColumnPart = FMT == GGUF_FMT_Q4K   ? 2048u
                                          : FMT == GGUF_FMT_Q6K ? GGUF_Q6K_SCALES
                                          : FMT == GGUF_FMT_Q5K ? GGUF_Q5K_META
                                          : FMT == GGUF_FMT_Q80 ? GGUF_Q80_SCALES
                                                                : GGUF_IQ4_SCALES;
  __device__ __forceinline__ void open(const uint8_t *record, uint32_t lane) {
    const uint4 *p = reinterpret_cast<const uint4 *>(record);
    mine = p + lane;
    column = p + kColumnPart / 16u + (lane & 15u);
    if constexpr (FMT == GGUF_FMT_Q6K) d = reinterpret_cast<const uint16_t *>(record + GGUF_Q6K_D) + (lane & 15u);
    if constexpr (FMT == GGUF_FMT_Q5K) fifth = reinterpret_cast<const uint2 *>(record + GGUF_Q5K_HIGH) + lane;
    if constexpr (FMT == GGUF_FMT_IQ4XS) meta8 = reinterpret_cast<const uint2 *>(record + GGUF_IQ4_SCALES) + (lane & 15u);
  }
  __device__ __forceinline__ void advance() {
    constexpr uint32_t kVectors = gguf_record_bytes(FMT) / 16u;
    mine += kVectors;
    column += kVectors;
    if constexpr (FMT == GGUF_FMT_Q6K) d += kVectors * 8u;
    if constexpr (FMT == GGUF_FMT_Q5K) fifth += kVectors * 2u;
    if constexpr (FMT == GGUF_FMT_IQ4XS) meta8 += kVectors * 2u;
  }
};

template <uint32_t FMT> struct Record;
template <> struct Record<GGUF_FMT_Q4K> {
  static constexpr uint32_t kLoads = 3;   // load_piece
  uint4 n0, n1, meta;
  __device__ __forceinline__ void load(const Cursor<GGUF_FMT_Q4K> &at) {
    n0 = load_stream(at.mine);
    n1 = load_stream(at.mine + 64);
    meta = load_stream(at.column);
  }
};
template <> struct Record<GGUF_FMT_Q6K> {
  static constexpr uint32_t kLoads = 5;   // load_piece
  uint4 n0, n1, high, scales;
  uint32_t d;
  __device__ __forceinline__ void load(const Cursor<GGUF_FMT_Q6K> &at) {
    n0 = load_stream(at.mine);
    n1 = load_stream(at.mine + 64);
    high = load_stream(at.mine + 128);
    scales = load_stream(at.column);
    d = __builtin_nontemporal_load(at.d);
  }
};

template <> struct Record<GGUF_FMT_Q5K> {
  static constexpr uint32_t kLoads = 4;   // load_piece
  uint4 n0, n1, meta;
  uint2 fifth;
  __device__ __forceinline__ void load(const Cursor<GGUF_FMT_Q5K> &at) {
    n0 = load_stream(at.mine);
    n1 = load_stream(at.mine + 64);
    meta = load_stream(at.column);
    fifth = *at.fifth;
  }
};
template <> struct Record<GGUF_FMT_Q80> {
  static constexpr uint32_t kLoads = 5;   // load_piece
  uint4 v[4], scales;
  __device__ __forceinline__ void load(const Cursor<GGUF_FMT_Q80> &at) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = load_stream(at.mine + 64 * i);
    scales = load_stream(at.column);
  }
};

template <> struct Record<GGUF_FMT_IQ4XS> {
  static constexpr uint32_t kLoads = 3;   // load_piece
  uint4 n0, n1;
  uint2 meta;  // x: d | scales_h << 16; y: the low four bits of the eight groups' scales
  __device__ __forceinline__ void load(const Cursor<GGUF_FMT_IQ4XS> &at) {
    n0 = load_stream(at.mine);
    n1 = load_stream(at.mine + 64);
    meta = *at.meta8;
  }
};
template <> struct Record<GGUF_FMT_IQ4NL> {
  static constexpr uint32_t kLoads = 3;   // load_piece
  uint4 n0, n1, scales;
  __device__ __forceinline__ void load(const Cursor<GGUF_FMT_IQ4NL> &at) {
    n0 = load_stream(at.mine);
    n1 = load_stream(at.mine + 64);
    scales = load_stream(at.column);
  }
};

// The eight groups' operand registers of a record, group g's in ops[g].
template <uint32_t FMT>
__device__ __forceinline__ void iq4_record_operands(const Record<FMT> &r, uint4 ops[8]) {
  ops[0] = iq4_operands(r.n0.x);
  ops[1] = iq4_operands(r.n0.y);
  ops[2] = iq4_operands(r.n0.z);
  ops[3] = iq4_operands(r.n0.w);
  ops[4] = iq4_operands(r.n1.x);
  ops[5] = iq4_operands(r.n1.y);
  ops[6] = iq4_operands(r.n1.z);
  ops[7] = iq4_operands(r.n1.w);
}
__device__ __forceinline__ void record_operands(const Record<GGUF_FMT_IQ4XS> &r, uint4 ops[8]) { iq4_record_operands(r, ops); }
__device__ __forceinline__ void record_operands(const Record<GGUF_FMT_IQ4NL> &r, uint4 ops[8]) { iq4_record_operands(r, ops); }
// Group g's scale of an IQ4_XS record's column: d * (ls - 32), ls its six bits of scales_l and scales_h (exact).
__device__ __forceinline__ float iq4xs_scale(const uint2 &meta, uint32_t g) {
  const uint32_t ls = ((meta.y >> (4u * g)) & 15u) | (((meta.x >> (16u + 2u * g)) & 3u) << 4);
  return half_bits_to_float(meta.x & 0xFFFFu) * float(int(ls) - 32);
}
__device__ __forceinline__ void record_operands(const Record<GGUF_FMT_Q5K> &r, uint4 ops[8]) {
  ops[0] = q5_operands<false, 0>(r.n0.x, r.n0.y, r.fifth.x);
  ops[1] = q5_operands<true, 4>(r.n0.x, r.n0.y, r.fifth.x);
  ops[2] = q5_operands<false, 8>(r.n0.z, r.n0.w, r.fifth.x);
  ops[3] = q5_operands<true, 12>(r.n0.z, r.n0.w, r.fifth.x);
  ops[4] = q5_operands<false, 0>(r.n1.x, r.n1.y, r.fifth.y);
  ops[5] = q5_operands<true, 4>(r.n1.x, r.n1.y, r.fifth.y);
  ops[6] = q5_operands<false, 8>(r.n1.z, r.n1.w, r.fifth.y);
  ops[7] = q5_operands<true, 12>(r.n1.z, r.n1.w, r.fifth.y);
}
__device__ __forceinline__ void record_operands(const Record<GGUF_FMT_Q80> &r, uint4 ops[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    ops[2 * i] = q8_operands(r.v[i].x, r.v[i].y);
    ops[2 * i + 1] = q8_operands(r.v[i].z, r.v[i].w);
  }
}
// Group g's fp16 scale of a Q8_0 record's column.
__device__ __forceinline__ float q8_scale(const uint4 &scales, uint32_t g) {
  const uint32_t word = g < 2 ? scales.x : g < 4 ? scales.y : g < 6 ? scales.z : scales.w;
  return half_bits_to_float((word >> (16u * (g & 1u))) & 0xFFFFu);
}
// Group g's scale of a record of one of the formats whose groups carry one scale and no minimum.
__device__ __forceinline__ float group_scale(const Record<GGUF_FMT_Q80> &r, uint32_t g) { return q8_scale(r.scales, g); }
__device__ __forceinline__ float group_scale(const Record<GGUF_FMT_IQ4NL> &r, uint32_t g) { return q8_scale(r.scales, g); }
__device__ __forceinline__ float group_scale(const Record<GGUF_FMT_IQ4XS> &r, uint32_t g) { return iq4xs_scale(r.meta, g); }
__device__ __forceinline__ void record_operands(const Record<GGUF_FMT_Q4K> &r, uint4 ops[8]) {
  ops[0] = q4_operands<false>(r.n0.x, r.n0.y);
  ops[1] = q4_operands<true>(r.n0.x, r.n0.y);
  ops[2] = q4_operands<false>(r.n0.z, r.n0.w);
  ops[3] = q4_operands<true>(r.n0.z, r.n0.w);
  ops[4] = q4_operands<false>(r.n1.x, r.n1.y);
  ops[5] = q4_operands<true>(r.n1.x, r.n1.y);
  ops[6] = q4_operands<false>(r.n1.z, r.n1.w);
  ops[7] = q4_operands<true>(r.n1.z, r.n1.w);
}
__device__ __forceinline__ void record_operands(const Record<GGUF_FMT_Q6K> &r, uint4 ops[8]) {
  ops[0] = q6_operands<false, 0>(r.n0.x, r.n0.y, r.high.x);
  ops[1] = q6_operands<true, 4>(r.n0.x, r.n0.y, r.high.x);
  ops[2] = q6_operands<false, 0>(r.n0.z, r.n0.w, r.high.y);
  ops[3] = q6_operands<true, 4>(r.n0.z, r.n0.w, r.high.y);
  ops[4] = q6_operands<false, 0>(r.n1.x, r.n1.y, r.high.z);
  ops[5] = q6_operands<true, 4>(r.n1.x, r.n1.y, r.high.z);
  ops[6] = q6_operands<false, 0>(r.n1.z, r.n1.w, r.high.w);
  ops[7] = q6_operands<true, 4>(r.n1.z, r.n1.w, r.high.w);
}

__device__ __forceinline__ float q6_scale(const uint4 &scales, uint32_t index) {
  const uint32_t word = index < 4 ? scales.x : index < 8 ? scales.y : index < 12 ? scales.z : scales.w;
  return float(int(int8_t((word >> (8u * (index & 3u))) & 0xFFu)));
}

// ---------------------------------------------------------------------------------------------
// Loads through buffer resources.
// ---------------------------------------------------------------------------------------------
// Streams are read through buffer resources: a load past the end of its range returns zeros and
// moves no memory, so the software pipeline below needs no branch around a load and no
// special case at the end of a range, and its address arithmetic is one 32-bit add per stream.
using Resource = __amdgpu_buffer_rsrc_t;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
__device__ __forceinline__ Resource make_resource(const void *base, uint32_t bytes) {
  // The base must be wave-uniform (it lives in scalar registers).
  const uint64_t v = reinterpret_cast<uint64_t>(base);
  // readfirstlane returns a signed int: widen each half as unsigned.
  const uint32_t hi = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v >> 32))));
  const uint32_t lo = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v))));
  const uint64_t u = (uint64_t(hi) << 32) | uint64_t(lo);
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(u), 0, __builtin_amdgcn_readfirstlane(int(bytes)), 0x00020000);
}
constexpr int kStreamOnce = 2;  // non-temporal: weights are read once
template <int Aux> __device__ __forceinline__ uint4 load128(Resource r, uint32_t offset) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, int(offset), 0, Aux);
  return make_uint4(v.x, v.y, v.z, v.w);
}
// Sixteen (four) bytes a lane of a wave, from memory straight into LDS (`to` the wave's first lane's, the others after it).
typedef __attribute__((address_space(3))) void LdsVoid;
template <uint32_t Bytes> __device__ __forceinline__ void load_to_lds(Resource r, uint32_t offset, void *to) {
  static_assert(Bytes == 16u || Bytes == 4u);
  if constexpr (Bytes == 16u) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LdsVoid *)to, 16, int(offset), 0, 0, 0);
  else __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LdsVoid *)to, 4, int(offset), 0, 0, 0);
}
// Vector-memory instructions that may be in flight behind a wait (s_waitcnt's vmcnt alone).
template <uint32_t N> __device__ __forceinline__ void wait_loads() {
  static_assert(N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((N & 15u) | ((N >> 4) << 14) | 0x0F70u);
}
// Piece I of a record's load, one vector-memory instruction each: Record::kLoads of them are a record, which is what the waits of
// a loop that counts its loads in flight rest on. `mine` is the lane's 16 bytes of the record's first 1024-byte part, `column`
// its column's scale field, both as byte offsets into the resource.
__device__ __forceinline__ uint32_t record_lane() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }
template <uint32_t I> __device__ __forceinline__ void load_piece(Record<GGUF_FMT_Q4K> &rec, Resource r, uint32_t mine, uint32_t column) {
  if constexpr (I == 0) rec.n0 = load128<kStreamOnce>(r, mine);
  else if constexpr (I == 1) rec.n1 = load128<kStreamOnce>(r, mine + 1024u);
  else rec.meta = load128<kStreamOnce>(r, column);
  static_assert(I < 3);
}
template <uint32_t I> __device__ __forceinline__ void load_piece(Record<GGUF_FMT_Q6K> &rec, Resource r, uint32_t mine, uint32_t column) {
  if constexpr (I == 0) rec.n0 = load128<kStreamOnce>(r, mine);
  else if constexpr (I == 1) rec.n1 = load128<kStreamOnce>(r, mine + 1024u);
  else if constexpr (I == 2) rec.high = load128<kStreamOnce>(r, mine + 2048u);
  else if constexpr (I == 3) rec.scales = load128<kStreamOnce>(r, column);
  else {
    // The lane's 16 l and the column's 16 c locate the record and c: d sits at record + 3328 + 2 c.
    const uint32_t lane = record_lane();
    rec.d = __builtin_amdgcn_raw_buffer_load_b16(r, int(mine - 16u * lane + GGUF_Q6K_D + 2u * (lane & 15u)), 0, kStreamOnce);
  }
  static_assert(I < 5);
}
template <uint32_t I> __device__ __forceinline__ void load_piece(Record<GGUF_FMT_Q5K> &rec, Resource r, uint32_t mine, uint32_t column) {
  if constexpr (I == 0) rec.n0 = load128<kStreamOnce>(r, mine);
  else if constexpr (I == 1) rec.n1 = load128<kStreamOnce>(r, mine + 1024u);
  else if constexpr (I == 2) rec.meta = load128<kStreamOnce>(r, column);
  else {
    // The lane's 8 bytes of fifth bits sit at record + 2048 + 8 l; `mine` is record + 16 l.
    const u32x2 fifth = __builtin_amdgcn_raw_buffer_load_b64(r, int(mine - 8u * record_lane() + GGUF_Q5K_HIGH), 0, kStreamOnce);
    rec.fifth = make_uint2(fifth.x, fifth.y);
  }
  static_assert(I < 4);
}
template <uint32_t I> __device__ __forceinline__ void load_piece(Record<GGUF_FMT_Q80> &rec, Resource r, uint32_t mine, uint32_t column) {
  if constexpr (I < 4) rec.v[I] = load128<kStreamOnce>(r, mine + 1024u * I);
  else rec.scales = load128<kStreamOnce>(r, column);
  static_assert(I < 5);
}
template <uint32_t I> __device__ __forceinline__ void load_piece(Record<GGUF_FMT_IQ4XS> &rec, Resource r, uint32_t mine, uint32_t) {
  if constexpr (I == 0) rec.n0 = load128<kStreamOnce>(r, mine);
  else if constexpr (I == 1) rec.n1 = load128<kStreamOnce>(r, mine + 1024u);
  else {
    // The column's 8 bytes sit at record + 2048 + 8 c; `mine` is record + 16 l.
    const uint32_t lane = record_lane();
    const u32x2 meta = __builtin_amdgcn_raw_buffer_load_b64(r, int(mine - 16u * lane + GGUF_IQ4_SCALES + 8u * (lane & 15u)), 0, kStreamOnce);
    rec.meta = make_uint2(meta.x, meta.y);
  }
  static_assert(I < 3);
}
template <uint32_t I> __device__ __forceinline__ void load_piece(Record<GGUF_FMT_IQ4NL> &rec, Resource r, uint32_t mine, uint32_t column) {
  if constexpr (I == 0) rec.n0 = load128<kStreamOnce>(r, mine);
  else if constexpr (I == 1) rec.n1 = load128<kStreamOnce>(r, mine + 1024u);
  else rec.scales = load128<kStreamOnce>(r, column);
  static_assert(I < 3);
}
template <uint32_t FMT> __device__ __forceinline__ void load_record(Record<FMT> &rec, Resource r, uint32_t mine, uint32_t column) {
  [&]<uint32_t... I>(std::integer_sequence<uint32_t, I...>) __attribute__((always_inline)) {
    (load_piece<I>(rec, r, mine, column), ...);
  }(std::make_integer_sequence<uint32_t, Record<FMT>::kLoads>{});
}

} // namespace splash::kernels
