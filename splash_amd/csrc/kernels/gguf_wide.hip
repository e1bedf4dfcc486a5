// The projections of a prompt chunk: many rows against a K-quant weight image (abi/Gguf.h), bound by the matrix cores.
//
// A 4-, 5- or 6-bit weight is d * (sc * code) - dmin * mn with an integer sc * code, which the decode kernels cannot use
// (their bf16 operands hold eight bits) and so multiply every group's sum by its scale on the vector ALU: an fp32
// multiply-add for every 32 products of an output, as long as the matrix cores take for them. fp16 holds eleven bits:
// sc * code is at most 63 * 31 and exact, so a whole super-block of 256 inputs accumulates in the matrix cores and costs
// an output one multiply-add by d, and the constant term one more MFMA against the rows' group sums and one by dmin. A
// Q6_K product needs twelve bits: it is the rounded fp16 product plus the exact fp16 remainder, two MFMAs. The rows
// enter as fp16 too, scaled by a power of two a row (the wide table), which keeps all eight bits of a bf16 value down to
// 2^-28 of its row's largest. The fp32 sums of 768 inputs lie 4 to 12 times closer to 64-bit ones than the decode kernels'.
//
// Split: a wave owns 32 columns (a record of two column tiles each super-block, dequantized once in its registers) of
// all of the workgroup's 128 rows, whose operands go from memory straight into LDS, three stages of two groups ahead of
// their use in four buffers, one barrier a stage. (Through registers, one stage ahead, which is what 256 of them leave
// room for, waves waited a quarter of their time: gate/up 1.27, the SwiGLU rows' projection 0.97 ms where it was 1.18 and
// 0.91; an expert's tiles, whose rows come from further away, 215 and 158 us where they take 192 and 149. A row
// tile's operands read two tiles ahead, or waves of a priority that follows the phase, changed nothing.) Two waves a SIMD
// overlap the conversion of one with the MFMAs of the other. At 2048 rows of the 5120 x 2 x 25600 Q4_K gate/up pair a
// launch takes 1.09 ms (985 TFLOP/s of the projection's own operations; the 64-row windows of the decode kernels took
// 2.38 ms), at 25600 x 5120 Q6_K 0.86 ms (2.2 ms): with the constant terms and the second product that is 1.11 and 1.25
// PFLOP/s of MFMAs, where a large fp16 library product of normally distributed values reaches 1.25 (of zeros 1.74: the card's
// power limits it). The matrix cores are busy 57 and 64 % of the cycles, a SIMD issues vector instructions in 60 and 54 %, and
// waves wait 14 to 15 %.
#include "abi/Gguf.h"
#include "abi/Moe.h"
#include "backend/KernelRegistry.hpp"
#include "kernels/gguf_records.hpp"
#include "kernels/gguf_wide_table.hpp"
#include <type_traits>
#include <utility>

namespace splash::kernels {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
__device__ __forceinline__ f16x2 as_f16x2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ f16x8 as_f16x8(uint4 v) { return __builtin_bit_cast(f16x8, v); }
__device__ __forceinline__ f16x2 both(float v) { return f16x2{_Float16(v), _Float16(v)}; }

// ---------------------------------------------------------------------------------------------
// The wide table.
// ---------------------------------------------------------------------------------------------
// A workgroup a row, straight to the table. The eight rows that share the table's 128-byte lines are neighbours on one die
// (workgroup b runs on die b % 8), so that its L2 writes whole lines.
template <bool Norm, uint32_t Held>
__device__ __forceinline__ void wide_table_row_out(const uint16_t *__restrict__ input, const uint16_t *__restrict__ weight, uint8_t *__restrict__ table,
                                                   const GgufWideTableParams &p, const uint32_t row, const uint32_t source) {
  uint4 *values = reinterpret_cast<uint4 *>(table + row / 16u * gguf_wide_tile_bytes(p.input_size)) + row % 16u;
  const float scale = wide_table_row<Norm, Held, 4>(input, weight, p, source, [&](uint32_t line, uint32_t, uint32_t, uint4 entry) __attribute__((always_inline)) {
    values[size_t(line) * 16u] = entry;
  });
  if (threadIdx.x == 0) wide_scales_of(table, p)[row] = scale;
}
template <bool Norm, uint32_t Held>
__global__ __launch_bounds__(256) void gguf_wide_table(const uint16_t *__restrict__ input, const uint16_t *__restrict__ weight,
                                                       uint8_t *__restrict__ table, GgufWideTableParams p) {
  const uint32_t row = wide_table_row_of(blockIdx.x);
  if (row < 16u * p.tiles) wide_table_row_out<Norm, Held>(input, weight, table, p, row, row);
}
// Where a row's table (abi/Gguf.h) has entry `kq` of operand `operand` of the super-block that `line` is of.
__device__ __forceinline__ uint4 *wide_row_entry(uint8_t *of, uint32_t inputSize, uint32_t line, uint32_t operand, uint32_t kq) {
  const uint32_t block = (line / 4u - operand) / GGUF_WIDE_OPERANDS;
  return reinterpret_cast<uint4 *>(of + (operand < 8u ? (block * 8u + operand) * 64u : inputSize * 2u + block * 64u) + 16u * kq);
}
// The rows' tables of rows as they are, a workgroup a row: whole lines of the row's own. (What the tables that a norm leaves are
// held against.)
__global__ __launch_bounds__(256) void gguf_wide_rows(const uint16_t *__restrict__ input, uint8_t *__restrict__ rows, GgufWideTableParams p) {
  const uint32_t row = blockIdx.x, bytes = gguf_wide_row_bytes(p.input_size);
  if (row >= p.rows) return;
  uint8_t *of = rows + size_t(row) * bytes;
  const float scale = wide_table_row<false, 4, 4>(input, nullptr, p, row, [&](uint32_t line, uint32_t operand, uint32_t kq, uint4 entry) __attribute__((always_inline)) {
    *wide_row_entry(of, p.input_size, line, operand, kq) = entry;
  });
  if (threadIdx.x == 0) reinterpret_cast<float *>(rows + size_t(p.rows) * bytes)[row] = scale;
}
// The normed rows as both: their wide table, and the rows' tables. With GGUF_WIDE_ROWS_NORM_RMS the rows' tables hold norm_rms's
// rows, whose sum of squares is added column by column: the experts' rows are the bits they are in every other path. Where that
// inverse is another float than the table's, the entries are made again. Bound by memory and a row's chain of sums; 2048 rows of
// 2048 inputs 10.8 us (8.8 without the flag, 7.0 the wide table alone, which norm_rms and gguf_wide_rows would follow with 8.4 and
// 4.9).
__global__ __launch_bounds__(256) void gguf_wide_table_norm_rows(const uint16_t *__restrict__ input, const uint16_t *__restrict__ weight,
                                                                 uint8_t *__restrict__ table, uint8_t *__restrict__ rows, GgufWideTableParams p) {
  constexpr uint32_t Held = 4;
  const uint32_t row = wide_table_row_of(blockIdx.x), bytes = gguf_wide_row_bytes(p.input_size);
  if (row >= 16u * p.tiles) return;
  __shared__ float scratch[16];
  const bool live = row < p.rows;
  const uint16_t *from = input + size_t(live ? row : 0u) * p.input_size;
  uint4 v[Held], w[Held], normed[Held];
  wide_row_load<Held, 4>(v, from, p.input_size, live);
  wide_row_load<Held, 4>(w, weight, p.input_size, live);
  const bool apart = live && (p.flags & GGUF_WIDE_ROWS_NORM_RMS);
  const float own = apart ? rms_inverse(from, p.input_size, scratch) : 0.f;
  const float inverse = wide_row_inverse(v, p.input_size, scratch + 4);
  const bool shared = live && (!apart || own == inverse);
  uint4 *values = reinterpret_cast<uint4 *>(table + row / 16u * gguf_wide_tile_bytes(p.input_size)) + row % 16u;
  uint8_t *of = rows + size_t(row) * bytes;
  float *rowScales = reinterpret_cast<float *>(rows + size_t(p.rows) * bytes);
  wide_row_norm(normed, v, w, inverse, p.input_size);
  const float scale = wide_row_entries<Held, 4>(normed, p.input_size, scratch + 8, [&](uint32_t line, uint32_t operand, uint32_t kq, uint4 entry) __attribute__((always_inline)) {
    values[size_t(line) * 16u] = entry;
    if (shared) *wide_row_entry(of, p.input_size, line, operand, kq) = entry;
  });
  if (threadIdx.x == 0) {
    wide_scales_of(table, p)[row] = scale;
    if (shared) rowScales[row] = scale;
  }
  if (shared || !live) return;
  wide_row_norm(normed, v, w, own, p.input_size);
  const float ownScale = wide_row_entries<Held, 4>(normed, p.input_size, scratch + 12, [&](uint32_t line, uint32_t operand, uint32_t kq, uint4 entry) __attribute__((always_inline)) {
    *wide_row_entry(of, p.input_size, line, operand, kq) = entry;
  });
  if (threadIdx.x == 0) rowScales[row] = ownScale;
}
// The table of a mixture's slots' own rows (or, Gathers, of the rows that they gather: row s is row slot_row[s] of the input;
// a chunk's gate/up pair gathers from the rows' tables instead, and this is what it is held against), zeros where the slot is
// empty, for the slots of the tiles there are.
template <bool Gathers>
__global__ __launch_bounds__(256) void gguf_wide_moe_table(const uint16_t *__restrict__ input, const uint32_t *__restrict__ slot_row,
                                                           const uint32_t *__restrict__ tile_total, uint8_t *__restrict__ table,
                                                           GgufWideTableParams p) {
  const uint32_t row = wide_table_row_of(blockIdx.x);
  if (row >= 16u * min(p.tiles, tile_total[0])) return;
  const uint32_t source = slot_row[row];
  wide_table_row_out<false, 4>(input, nullptr, table, p, row, Gathers || source == MOE_NO_ROW ? source : row);
}
// The same of up to GGUF_WIDE_TILE_INPUTS inputs, grid (tiles), 1024 threads: a tile a workgroup, a wave a row, the tile put
// together in LDS and written as it lies there. A row's own stores are 16 bytes each to a line of its own, 64 lines a wave's
// store; the tile's are 1 KB. In LDS a line's sixteen places are turned by its number, or the lanes of a row's store would all
// meet in the same four banks. 16384 slots and what fills their tiles: 2048 gathered inputs 32.5 us by the row, 34.1 by a wave
// a row without the tile, 28.1 so (5 TB/s of rows read and tables written); 768 of the slots' own 24.3, 16.9 and 16.1.
// Up to 2048 inputs, of which two workgroups fit a compute unit: with LDS for 4096 (144 KB, one a unit) 17408 gathered slots
// took 35.7 us of 2048 inputs (27.2 so), 43.2 of 2304 and 64.4 of 4096 where the rows' kernel takes 35.8 and 56.7. (4096 slots
// of 2304 11.4 for 12.2; the slots' own rows past 3072 inputs, 17408 of 3584, 58 for 84: not built for.)
template <bool Gathers>
__global__ __launch_bounds__(1024) void gguf_wide_moe_tile(const uint16_t *__restrict__ input, const uint32_t *__restrict__ slot_row,
                                                           const uint32_t *__restrict__ tile_total, uint8_t *__restrict__ table,
                                                           GgufWideTableParams p) {
  __shared__ __align__(16) uint4 staged[GGUF_WIDE_TILE_INPUTS / 256u * GGUF_WIDE_OPERANDS * 64u];
  const uint32_t tile = blockIdx.x, r = threadIdx.x >> 6, row = 16u * tile + r;
  if (tile >= min(p.tiles, tile_total[0])) return;
  auto turned = [](uint32_t place, uint32_t operand, uint32_t kq) __attribute__((always_inline)) { return place ^ ((4u * operand + kq) & 15u); };
  const uint32_t source = slot_row[row];
  const float scale = wide_table_row<false, GGUF_WIDE_TILE_INPUTS / 512u, 1>(
      input, nullptr, p, Gathers || source == MOE_NO_ROW ? source : row,
      [&](uint32_t line, uint32_t operand, uint32_t kq, uint4 entry) __attribute__((always_inline)) { staged[line * 16u + turned(r, operand, kq)] = entry; });
  if ((threadIdx.x & 63u) == 0) wide_scales_of(table, p)[row] = scale;
  __syncthreads();
  uint4 *values = reinterpret_cast<uint4 *>(table + tile * gguf_wide_tile_bytes(p.input_size));
  const uint32_t entries = p.input_size / 256u * GGUF_WIDE_OPERANDS * 64u;
  for (uint32_t e = threadIdx.x; e < entries; e += 1024u)
    values[e] = staged[(e & ~15u) | turned(e & 15u, (e >> 6) % GGUF_WIDE_OPERANDS, (e >> 4) & 3u)];
}
SP_REGISTER_KERNEL("gguf_wide_moe_gather_tile", &gguf_wide_moe_tile<true>);
SP_REGISTER_KERNEL("gguf_wide_moe_rows_tile", &gguf_wide_moe_tile<false>);
SP_REGISTER_KERNEL("gguf_wide_moe_gather", &gguf_wide_moe_table<true>);
SP_REGISTER_KERNEL("gguf_wide_moe_rows", &gguf_wide_moe_table<false>);
SP_REGISTER_KERNEL("gguf_wide_table", (&gguf_wide_table<false, 4>));
SP_REGISTER_KERNEL("gguf_wide_table_long", (&gguf_wide_table<false, 16>));
SP_REGISTER_KERNEL("gguf_wide_table_norm", (&gguf_wide_table<true, 4>));
SP_REGISTER_KERNEL("gguf_wide_rows", &gguf_wide_rows);
SP_REGISTER_KERNEL("gguf_wide_table_norm_rows", &gguf_wide_table_norm_rows);

// ---------------------------------------------------------------------------------------------
// The wide projection.
// ---------------------------------------------------------------------------------------------
#define GGUF_WIDE_PLAIN 0u
#define GGUF_WIDE_RESIDUAL 1u
#define GGUF_WIDE_GATE_UP 2u
#define GGUF_WIDE_PARTIAL 3u

// A record as it passes through a wave: half of its nibbles at a time, what they share with the other half kept.
template <uint32_t FMT> struct WideRecord {
  uint4 codes[2];     // the nibbles of stages 0 and 1, of stages 2 and 3
  uint4 meta;         // Q4_K, Q5_K: d, dmin and the packed scales; Q6_K: the scales
  uint4 high;         // Q6_K: the high bits
  uint2 fifth;        // Q5_K: the fifth bits
  uint32_t d;         // Q6_K
};
// The loads of a record in three parts: what its first two stages need (and what all share), the codes of its last two, and
// the bits its last stage reads too. A part's count is the loop that issues it and what the waits for the rows count by: a
// load is one vector-memory instruction.
template <uint32_t FMT> constexpr uint32_t kWideFirstLoads = FMT == GGUF_FMT_Q6K ? 3u : 2u;
template <uint32_t FMT> constexpr uint32_t kWideSecondLoads = 1u;
template <uint32_t FMT> constexpr uint32_t kWideLateLoads = FMT == GGUF_FMT_Q4K ? 0u : 1u;
template <uint32_t N, typename F> __device__ __forceinline__ void each_load(F &&load) {
  [&]<uint32_t... I>(std::integer_sequence<uint32_t, I...>) __attribute__((always_inline)) {
    (load(std::integral_constant<uint32_t, I>{}), ...);
  }(std::make_integer_sequence<uint32_t, N>{});
}
template <uint32_t FMT> __device__ __forceinline__ void load_first(WideRecord<FMT> &rec, Resource r, uint32_t mine, uint32_t lane) {
  const uint32_t record = mine - 16u * lane, c = lane & 15u;
  each_load<kWideFirstLoads<FMT>>([&](auto i) __attribute__((always_inline)) {
    if constexpr (i == 0u) rec.codes[0] = load128<kStreamOnce>(r, mine);
    else if constexpr (i == 1u) rec.meta = load128<kStreamOnce>(r, record + Cursor<FMT>::kColumnPart + 16u * c);
    else {
      static_assert(i == 2u && FMT == GGUF_FMT_Q6K);
      rec.d = __builtin_amdgcn_raw_buffer_load_b16(r, int(record + GGUF_Q6K_D + 2u * c), 0, kStreamOnce);
    }
  });
}
template <uint32_t FMT> __device__ __forceinline__ void load_second(WideRecord<FMT> &rec, Resource r, uint32_t mine) {
  each_load<kWideSecondLoads<FMT>>([&](auto i) __attribute__((always_inline)) {
    static_assert(i == 0u);
    rec.codes[1] = load128<kStreamOnce>(r, mine + 1024u);
  });
}
template <uint32_t FMT> __device__ __forceinline__ void load_late(WideRecord<FMT> &rec, Resource r, uint32_t mine, uint32_t lane) {
  each_load<kWideLateLoads<FMT>>([&](auto i) __attribute__((always_inline)) {
    static_assert(i == 0u && (FMT == GGUF_FMT_Q6K || FMT == GGUF_FMT_Q5K));
    if constexpr (FMT == GGUF_FMT_Q6K) rec.high = load128<kStreamOnce>(r, mine + GGUF_Q6K_HIGH);
    else {
      const u32x2 fifth = __builtin_amdgcn_raw_buffer_load_b64(r, int(mine - 8u * lane + GGUF_Q5K_HIGH), 0, kStreamOnce);
      rec.fifth = make_uint2(fifth.x, fifth.y);
    }
  });
}
// What its operands need of `meta` once a super-block.
template <uint32_t FMT> struct WideScales {
  float d, dmin;
  uint32_t sc_lo, sc_hi, mn_lo, mn_hi;   // Q6_K: the sixteen signed scales
};
__device__ __forceinline__ uint32_t byte_pair(uint32_t word, uint32_t first, uint32_t second) {   // fp16 1024 + byte, of two bytes
  return __builtin_amdgcn_perm(0x64646464u, word, 0x04000400u | first | (second << 16));
}
template <uint32_t FMT> __device__ __forceinline__ WideScales<FMT> wide_scales(const WideRecord<FMT> &rec) {
  if constexpr (FMT == GGUF_FMT_Q6K) {
    // signed bytes: byte ^ 0x80 is scale + 128
    return {half_bits_to_float(rec.d), 0.f, rec.meta.x ^ 0x80808080u, rec.meta.y ^ 0x80808080u, rec.meta.z ^ 0x80808080u, rec.meta.w ^ 0x80808080u};
  } else {
    const Q4KScales q = q4k_scales(rec.meta);
    return {q.d, -32.f * q.dmin, q.sc_lo, q.sc_hi, q.mn_lo, q.mn_hi};   // (the sums are stored divided by 32)
  }
}
// The mins of the eight groups as fp16: the constant term's operand.
template <uint32_t FMT> __device__ __forceinline__ uint4 wide_mins(const WideScales<FMT> &s) {
  const f16x2 k = both(1024.f);
  return make_uint4(as_word(as_f16x2(byte_pair(s.mn_lo, 0, 1)) - k), as_word(as_f16x2(byte_pair(s.mn_lo, 2, 3)) - k),
                    as_word(as_f16x2(byte_pair(s.mn_hi, 0, 1)) - k), as_word(as_f16x2(byte_pair(s.mn_hi, 2, 3)) - k));
}
// Groups 2 S and 2 S + 1 of a record: sc * code as fp16 (Q6_K: rounded, and what the rounding left).
template <uint32_t FMT> struct WideOperands {
  uint4 high[2];
  uint4 low[FMT == GGUF_FMT_Q6K ? 2 : 1];
};
template <uint32_t FMT, uint32_t S>
__device__ __forceinline__ WideOperands<FMT> wide_operands(const WideRecord<FMT> &rec, const WideScales<FMT> &sc) {
  WideOperands<FMT> out;
  const uint4 n = rec.codes[S >> 1];
  const uint32_t wa = S & 1u ? n.z : n.x, wb = S & 1u ? n.w : n.y;
  if constexpr (FMT == GGUF_FMT_Q4K) {
    // a nibble at bits 0..3 is 1024 + code under fp16's 2^10, one at bits 4..7 is 64 + code under 2^6
    const uint32_t words[4] = {wa, wa >> 8, wb, wb >> 8};
    const uint32_t word = S < 2 ? sc.sc_lo : sc.sc_hi;
    const f16x2 first = as_f16x2(byte_pair(word, (2u * S) & 3u, (2u * S) & 3u)) - both(1024.f);
    const f16x2 second = as_f16x2(byte_pair(word, (2u * S + 1u) & 3u, (2u * S + 1u) & 3u)) - both(1024.f);
    const f16x2 firstOff = first * both(-1024.f), secondOff = second * both(-64.f);
    uint32_t a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a[i] = as_word(__builtin_elementwise_fma(as_f16x2(and_or(words[i], 0x000F000Fu, 0x64006400u)), first, firstOff));
      b[i] = as_word(__builtin_elementwise_fma(as_f16x2(and_or(words[i], 0x00F000F0u, 0x54005400u)), second, secondOff));
    }
    out.high[0] = make_uint4(a[0], a[1], a[2], a[3]);
    out.high[1] = make_uint4(b[0], b[1], b[2], b[3]);
  } else if constexpr (FMT == GGUF_FMT_Q5K) {
    const uint32_t fifth = S < 2 ? rec.fifth.x : rec.fifth.y;
    const uint4 code[2] = {q5_operands<false, 8u * (S & 1u), 0x64006400u>(wa, wb, fifth), q5_operands<true, 8u * (S & 1u) + 4u, 0x64006400u>(wa, wb, fifth)};
    const uint32_t word = S < 2 ? sc.sc_lo : sc.sc_hi;
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
      const f16x2 scale = as_f16x2(byte_pair(word, (2u * S + i) & 3u, (2u * S + i) & 3u)) - both(1024.f), off = scale * both(-1024.f);
      const uint32_t words[4] = {code[i].x, code[i].y, code[i].z, code[i].w};
      uint32_t a[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = as_word(__builtin_elementwise_fma(as_f16x2(words[e]), scale, off));
      out.high[i] = make_uint4(a[0], a[1], a[2], a[3]);
    }
  } else {
    const uint32_t hw = S == 0 ? rec.high.x : S == 1 ? rec.high.y : S == 2 ? rec.high.z : rec.high.w;
    const uint4 code[2] = {q6_operands<false, 0, 0x64006400u>(wa, wb, hw), q6_operands<true, 4, 0x64006400u>(wa, wb, hw)};
    const uint32_t word = S == 0 ? sc.sc_lo : S == 1 ? sc.sc_hi : S == 2 ? sc.mn_lo : sc.mn_hi;   // of the four 16-input blocks
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
      const uint32_t words[4] = {code[i].x, code[i].y, code[i].z, code[i].w};
      uint32_t a[4], b[4];
#pragma unroll
      for (uint32_t e = 0; e < 4; ++e) {
        const uint32_t block = 2u * i + (e >> 1);
        const f16x2 scale = as_f16x2(byte_pair(word, block, block)) - both(1152.f);
        const f16x2 value = as_f16x2(words[e]) - both(1056.f);   // code - 32
        const f16x2 product = value * scale;
        a[e] = as_word(product);
        b[e] = as_word(__builtin_elementwise_fma(value, scale, -product));   // exact: an integer below the product's last bit
      }
      out.high[i] = make_uint4(a[0], a[1], a[2], a[3]);
      out.low[i] = make_uint4(b[0], b[1], b[2], b[3]);
    }
  }
  return out;
}

// The same groups' weights rounded once to half: the staged rule (gguf_linear.hip), whole values that need no scale after.
template <uint32_t FMT, uint32_t S>
__device__ __forceinline__ WideOperands<FMT> wide_staged_operands(const WideRecord<FMT> &rec, const WideScales<FMT> &sc) {
  WideOperands<FMT> out{};
  const uint4 n = rec.codes[S >> 1];
  const uint32_t wa = S & 1u ? n.z : n.x, wb = S & 1u ? n.w : n.y;
  uint4 code[2];
  if constexpr (FMT == GGUF_FMT_Q4K) {
    code[0] = q4_operands<false, 0x64006400u>(wa, wb);
    code[1] = q4_operands<true, 0x64006400u>(wa, wb);
  } else if constexpr (FMT == GGUF_FMT_Q5K) {
    const uint32_t fifth = S < 2 ? rec.fifth.x : rec.fifth.y;
    code[0] = q5_operands<false, 8u * (S & 1u), 0x64006400u>(wa, wb, fifth);
    code[1] = q5_operands<true, 8u * (S & 1u) + 4u, 0x64006400u>(wa, wb, fifth);
  } else {
    const uint32_t hw = S == 0 ? rec.high.x : S == 1 ? rec.high.y : S == 2 ? rec.high.z : rec.high.w;
    code[0] = q6_operands<false, 0, 0x64006400u>(wa, wb, hw);
    code[1] = q6_operands<true, 4, 0x64006400u>(wa, wb, hw);
  }
#pragma unroll
  for (uint32_t i = 0; i < 2; ++i) {
    const uint32_t words[4] = {code[i].x, code[i].y, code[i].z, code[i].w};
    uint32_t a[4];
#pragma unroll
    for (uint32_t e = 0; e < 4; ++e) {
      f16x2 half;
      if constexpr (FMT == GGUF_FMT_Q6K) {
        const uint32_t word = S == 0 ? sc.sc_lo : S == 1 ? sc.sc_hi : S == 2 ? sc.mn_lo : sc.mn_hi;
        const f16x2 value = as_f16x2(words[e]) - both(1056.f);
        const float s = sc.d * (byte_of(word, 2u * i + (e >> 1)) - 128.f);
        half = f16x2{_Float16(s * float(value.x)), _Float16(s * float(value.y))};
      } else {
        const uint32_t g = 2u * S + i;
        const f16x2 value = as_f16x2(words[e]) - both(1024.f);
        const float s = sc.d * byte_of(g < 4 ? sc.sc_lo : sc.sc_hi, g & 3u), m = 0.03125f * sc.dmin * byte_of(g < 4 ? sc.mn_lo : sc.mn_hi, g & 3u);
        half = f16x2{_Float16(__fmaf_rn(s, float(value.x), m)), _Float16(__fmaf_rn(s, float(value.y), m))};
      }
      a[e] = as_word(half);
    }
    out.high[i] = make_uint4(a[0], a[1], a[2], a[3]);
  }
  return out;
}

// What a workgroup computes: its wave's two column tiles (image null: a tile past the last), its row tiles, its part of K.
struct WideTile {
  const uint8_t *image[2];
  uint32_t column[2];
  uint32_t tile0, tilesHere, rows;   // rows: those of the output
  uint32_t b0, count, split;
};
// The two column tiles of wave `wave` of column group `group`: neighbours, or of a gate/up pair the same columns of both.
template <uint32_t FMT, bool GateUp>
__device__ __forceinline__ void wide_columns(WideTile &w, const uint8_t *seg0, const uint8_t *seg1, const uint8_t *seg2, const GgufWideParams &p,
                                             uint32_t group, uint32_t wave) {
  const uint64_t tileBytes = uint64_t(p.input_size / GGUF_BLOCK) * gguf_record_bytes(FMT);
  if constexpr (GateUp) {
    const uint32_t tile = group * 4u + wave;
    const bool live = tile * 16u < p.cols[0];
    w.image[0] = live ? seg0 + tile * tileBytes : nullptr;
    w.image[1] = live ? seg1 + tile * tileBytes : nullptr;
    w.column[0] = w.column[1] = p.offset[0] + tile * 16u;
  } else {
    const uint8_t *seg = seg0;
    uint32_t offset = p.offset[0], columns = p.cols[0];
    const uint32_t first = (p.cols[0] + GGUF_WIDE_COLUMNS - 1u) / GGUF_WIDE_COLUMNS, second = (p.cols[1] + GGUF_WIDE_COLUMNS - 1u) / GGUF_WIDE_COLUMNS;
    if (group >= first) {
      group -= first;
      seg = seg1;
      offset = p.offset[1];
      columns = p.cols[1];
      if (group >= second) {
        group -= second;
        seg = seg2;
        offset = p.offset[2];
        columns = p.cols[2];
      }
    }
#pragma unroll
    for (uint32_t r = 0; r < 2; ++r) {
      const uint32_t tile = group * 8u + wave * 2u + r;
      w.image[r] = tile * 16u < columns ? seg + tile * tileBytes : nullptr;
      w.column[r] = offset + tile * 16u;
    }
  }
}

// A workgroup's LDS: a super-block's four stages, each [row tile][group][lane], and its sums. Objects of their own, so that a
// read of one does not wait for what is on its way into another.
struct WideLds {
  uint4 *rows0, *rows1, *rows2, *rows3, *sums;
  f32x4 *scales;   // the row tiles' scales, four rows a vector
};
template <uint32_t T> constexpr uint32_t kWideScales = (T + 3) / 4 * 16;
template <uint32_t T> constexpr uint32_t kWideStageVectors = (T + 1) / 2 * 2 * 2 * 64;
template <uint32_t FMT, uint32_t T, bool Staged> constexpr uint32_t kWideSumVectors = FMT != GGUF_FMT_Q6K && !Staged ? (T + 3) / 4 * 4 * 64 : 1;

// Two neighbouring columns in memory, aligned as one is.
typedef uint32_t __attribute__((aligned(2), may_alias)) PairBits;
typedef float __attribute__((ext_vector_type(2), aligned(4), may_alias)) PairFloats;
// T: the row tiles a workgroup computes, at least those it takes (a tile past them multiplies zeros). Gathers: `table` holds
// the rows' tables (of p.rows rows), and slot s is row slot_row[s]. Eight neighbouring lanes fetch a line of a row, both
// groups of a stage; in LDS the row's eight places are turned by half the row's number, so that the sixteen rows that a
// quarter of the wave reads lie in all the banks.
template <uint32_t FMT, uint32_t EP, uint32_t T, bool Staged, bool Gathers = false>
__device__ __forceinline__ void wide_workgroup(const WideLds lds, const WideTile &w, const uint8_t *__restrict__ table, void *__restrict__ out,
                                               const uint16_t *__restrict__ residual, const GgufWideParams &p,
                                               const uint32_t *__restrict__ slot_row = nullptr) {
  constexpr uint32_t kRecord = gguf_record_bytes(FMT);
  constexpr bool kSums = FMT != GGUF_FMT_Q6K && !Staged, kTwice = FMT == GGUF_FMT_Q6K && !Staged, kGateUp = EP == GGUF_WIDE_GATE_UP;
  const uint32_t lane = threadIdx.x & 63u, c = lane & 15u, kq = lane >> 4;
  const uint32_t tile0 = w.tile0, tilesHere = w.tilesHere, b0 = w.b0, count = w.count, split = w.split;
  const uint32_t column[2] = {w.column[0], w.column[1]};
  Resource weights[2];
#pragma unroll
  for (uint32_t r = 0; r < 2; ++r)
    weights[r] = make_resource(w.image[r] ? w.image[r] + size_t(b0) * kRecord : table, w.image[r] ? count * kRecord : 0u);
  const uint32_t tileBytes = uint32_t(gguf_wide_tile_bytes(p.input_size));
  // (row tiles past the workgroup's, and super-blocks past its range, read as zeros or are not used)
  const uint32_t rowBytes = gguf_wide_row_bytes(p.input_size);
  const Resource rowValues = Gathers ? make_resource(table, p.rows * rowBytes) : make_resource(table + size_t(tile0) * tileBytes, tilesHere * tileBytes);

  f32x4 acc[2][T], dot[2][T];
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (uint32_t r = 0; r < 2; ++r)
#pragma unroll
    for (uint32_t t = 0; t < T; ++t) acc[r][t] = dot[r][t] = zero;

  // Stage n holds groups 2 (n % 4), 2 (n % 4) + 1 of super-block n / 4 (and with a super-block's last, its sums): this
  // wave's share of it, four (six) kilobytes, on its way into LDS three stages ahead of its use.
  constexpr uint32_t kShare = (T + 1) / 2, kSumShare = kSums ? (T + 3) / 4 : 0;
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
  const uint32_t mineAt = (threadIdx.x >> 7) * tileBytes + (threadIdx.x & 127u) * 16u;
  const uint32_t sumsAt = (threadIdx.x >> 6) * tileBytes + lane * 16u;
  // Of gathered rows: where this lane's row begins, a share's tiles; past every row for an empty slot, which reads as zeros.
  constexpr uint32_t kNowhere = 0xC0000000u;
  uint32_t rowAt[Gathers ? kShare : 1], rowSumsAt[Gathers && kSums ? kSumShare : 1], scaleAt = 0;
  if constexpr (Gathers) {
    auto sourceOf = [&](uint32_t tile, uint32_t r) __attribute__((always_inline)) {
      const uint32_t source = slot_row[16u * (tile0 + min(tile, tilesHere - 1u)) + r];
      return tile < tilesHere ? source : MOE_NO_ROW;
    };
    const uint32_t r = (threadIdx.x & 127u) >> 3, piece = (threadIdx.x & 7u) ^ (r >> 1), sumRow = lane >> 2, sumPiece = (lane & 3u) ^ (sumRow >> 2);
#pragma unroll
    for (uint32_t i = 0; i < kShare; ++i) {
      const uint32_t source = sourceOf(2u * i + (threadIdx.x >> 7), r);
      rowAt[i] = source < p.rows ? source * rowBytes + 16u * piece : kNowhere;
    }
    if constexpr (kSums) {
#pragma unroll
      for (uint32_t i = 0; i < kSumShare; ++i) {
        const uint32_t source = sourceOf(4u * i + wave, sumRow);
        rowSumsAt[i] = source < p.rows ? source * rowBytes + p.input_size * 2u + 16u * sumPiece : kNowhere;
      }
    }
    const uint32_t source = sourceOf(threadIdx.x >> 4, threadIdx.x & 15u);
    scaleAt = source < p.rows ? source * 4u : kNowhere;
  }
  auto stageRows = [&](auto stageConstant) __attribute__((always_inline)) -> uint4 * {
    constexpr uint32_t S = decltype(stageConstant)::value;
    return S == 0 ? lds.rows0 : S == 1 ? lds.rows1 : S == 2 ? lds.rows2 : lds.rows3;
  };
  auto fetch = [&](uint32_t block, auto stageConstant) __attribute__((always_inline)) {   // block counts from b0
    constexpr uint32_t S = decltype(stageConstant)::value;
    uint4 *to = stageRows(stageConstant) + 64u * wave;
    // (past the part of K: zeros, no traffic)
    if constexpr (Gathers) {
      const uint32_t past = block < count ? 0u : 0x80000000u;
#pragma unroll
      for (uint32_t i = 0; i < kShare; ++i) load_to_lds<16>(rowValues, rowAt[i] + (past + (b0 + block) * 512u + S * 128u), to + 256u * i);
      if constexpr (S == 3u && kSums) {
#pragma unroll
        for (uint32_t i = 0; i < kSumShare; ++i) load_to_lds<16>(rowValues, rowSumsAt[i] + (past + (b0 + block) * 64u), lds.sums + 64u * wave + 256u * i);
      }
      return;
    }
    const uint32_t at = block < count ? (b0 + block) * (GGUF_WIDE_OPERANDS * 1024u) + S * 2048u : 0x80000000u;
#pragma unroll
    for (uint32_t i = 0; i < kShare; ++i) load_to_lds<16>(rowValues, mineAt + (at + 2u * i * tileBytes), to + 256u * i);
    if constexpr (S == 3u) {
#pragma unroll
      for (uint32_t i = 0; i < kSumShare; ++i) load_to_lds<16>(rowValues, sumsAt + (at + 2048u + 4u * i * tileBytes), lds.sums + 64u * wave + 256u * i);
    }
  };
  // A record's first half (and what both share) is fetched two stages ahead of its use, and so is its second.
  WideRecord<FMT> rec[2];
  uint32_t mine = 16u * lane;   // of the next super-block to fetch
  auto fetchFirst = [&] {
#pragma unroll
    for (uint32_t r = 0; r < 2; ++r) load_first<FMT>(rec[r], weights[r], mine, lane);
  };
  auto fetchLate = [&] {
#pragma unroll
    for (uint32_t r = 0; r < 2; ++r) load_late<FMT>(rec[r], weights[r], mine, lane);
  };
  auto fetchSecond = [&] {
#pragma unroll
    for (uint32_t r = 0; r < 2; ++r) load_second<FMT>(rec[r], weights[r], mine);
    mine += kRecord;
  };
  // What a stage's loads are: its rows' (three stages ahead), then the weights'. A stage's rows are there when at most what
  // was asked for after them is on its way. (Counted by what issues them: the parts' own counts, of the lane's two records.)
  constexpr auto weightLoads = [](uint32_t stage) constexpr {
    return 2u * (stage == 0 ? kWideSecondLoads<FMT> : stage == 2u ? kWideFirstLoads<FMT> : stage == 3u ? kWideLateLoads<FMT> : 0u);
  };
  constexpr auto rowLoads = [](uint32_t stage) constexpr { return kShare + (stage == 3u ? kSumShare : 0u); };
  // (first of all loads, so that the first stage's wait and barrier are these's too)
  if (Gathers && wave < kWideScales<T> / 16u)
    load_to_lds<4>(make_resource(table + size_t(p.rows) * rowBytes, p.rows * 4u), scaleAt, lds.scales + 16u * wave);
  if (!Gathers && wave < kWideScales<T> / 16u)
    load_to_lds<4>(make_resource(table + gguf_wide_scales_offset(p.input_size, p.tiles) + tile0 * 64u, tilesHere * 64u), threadIdx.x * 4u,
                   lds.scales + 16u * wave);
  __builtin_amdgcn_sched_barrier(0);
  // (the loads before the first stage in the order of the stages that would have asked for them)
  fetch(0, std::integral_constant<uint32_t, 0>{});
  __builtin_amdgcn_sched_barrier(0);
  fetch(0, std::integral_constant<uint32_t, 1>{});
  __builtin_amdgcn_sched_barrier(0);
  fetchFirst();
  __builtin_amdgcn_sched_barrier(0);
  fetch(0, std::integral_constant<uint32_t, 2>{});
  __builtin_amdgcn_sched_barrier(0);
  fetchLate();
  __builtin_amdgcn_sched_barrier(0);
  for (uint32_t block = 0; block < count; ++block) {
    WideScales<FMT> scales[2];
#pragma unroll
    for (uint32_t r = 0; r < 2; ++r) scales[r] = wide_scales(rec[r]);
    auto run = [&](auto stageConstant) {
      constexpr uint32_t S = decltype(stageConstant)::value;
      // (behind stage S's rows: the weights of that stage and the two after it, and the two stages' rows between)
      wait_loads<weightLoads((S + 1u) & 3u) + rowLoads((S + 1u) & 3u) + weightLoads((S + 2u) & 3u) + rowLoads((S + 2u) & 3u) + weightLoads((S + 3u) & 3u)>();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      fetch(block + (S >= 1u ? 1u : 0u), std::integral_constant<uint32_t, (S + 3u) & 3u>{});
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (S == 0) fetchSecond();
      if constexpr (S == 2u) fetchFirst();
      __builtin_amdgcn_sched_barrier(0);
      const uint4 *rows = stageRows(stageConstant);
      WideOperands<FMT> operands[2];
#pragma unroll
      for (uint32_t r = 0; r < 2; ++r) {
        if constexpr (Staged) operands[r] = wide_staged_operands<FMT, S>(rec[r], scales[r]);
        else operands[r] = wide_operands<FMT, S>(rec[r], scales[r]);
      }
      uint4 mins[2];
      if constexpr (S == 3u && kSums) {
#pragma unroll
        for (uint32_t r = 0; r < 2; ++r) mins[r] = wide_mins(scales[r]);
      }
      if constexpr (S == 3u) fetchLate();   // (over the bits that the last operands were made of)
      // A row tile's operands leave LDS while the tile before it is multiplied.
      constexpr uint32_t kReads = S == 3u && kSums ? 3u : 2u;
      f16x8 a[2][3];
      auto read = [&](uint32_t t) {
#pragma unroll
        for (uint32_t g = 0; g < 2; ++g) a[t & 1u][g] = as_f16x8(rows[t * 128u + (Gathers ? 8u * c + ((4u * g + kq) ^ (c >> 1)) : g * 64u + lane)]);
        if constexpr (kReads == 3u) a[t & 1u][2] = as_f16x8(lds.sums[t * 64u + (Gathers ? 4u * c + (kq ^ (c >> 2)) : lane)]);
      };
      read(0);
#pragma unroll
      for (uint32_t t = 0; t < T; ++t) {
        if (t + 1 < T) read(t + 1);
#pragma unroll
        for (uint32_t g = 0; g < 2; ++g) {
#pragma unroll
          for (uint32_t r = 0; r < 2; ++r)
            dot[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t & 1u][g], as_f16x8(operands[r].high[g]), !Staged && S == 0 && g == 0 ? zero : dot[r][t], 0, 0, 0);
          if constexpr (kTwice) {
#pragma unroll
            for (uint32_t r = 0; r < 2; ++r) dot[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t & 1u][g], as_f16x8(operands[r].low[g]), dot[r][t], 0, 0, 0);
          }
        }
        if constexpr (S == 3u && !Staged) {
          f32x4 least[2];
          if constexpr (kSums) {
#pragma unroll
            for (uint32_t r = 0; r < 2; ++r) least[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t & 1u][2], as_f16x8(mins[r]), zero, 0, 0, 0);
          }
#pragma unroll
          for (uint32_t r = 0; r < 2; ++r)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              acc[r][t][v] = __fmaf_rn(dot[r][t][v], scales[r].d, acc[r][t][v]);
              if constexpr (kSums) acc[r][t][v] = __fmaf_rn(least[r][v], scales[r].dmin, acc[r][t][v]);
            }
        }
      }
      constexpr uint32_t kProducts = (kTwice ? 8u : 4u) + (S == 3u && kSums ? 2u : 0u);
      __builtin_amdgcn_sched_group_barrier(0x100, kReads, 0);
#pragma unroll
      for (uint32_t t = 0; t < T; ++t) {
        if (t + 1 < T) __builtin_amdgcn_sched_group_barrier(0x100, kReads, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, kProducts, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    run(std::integral_constant<uint32_t, 0>{});
    run(std::integral_constant<uint32_t, 1>{});
    run(std::integral_constant<uint32_t, 2>{});
    run(std::integral_constant<uint32_t, 3>{});
  }
  if constexpr (Staged) {
#pragma unroll
    for (uint32_t r = 0; r < 2; ++r)
#pragma unroll
      for (uint32_t t = 0; t < T; ++t) acc[r][t] = dot[r][t];
  }
  wait_loads<0>();   // (nothing is on its way into LDS when the workgroup gives it up)
  // Element (t, v) of this lane is row 16 (tile0 + t) + 4 kq + v, column column[r] + c. Neighbouring lanes trade one of every
  // two rows, so that a lane stores two columns of a row: half the stores, of twice the bytes. What a residual adds leaves
  // memory for all of the tiles at once. (The scales were loaded here, a row's behind the test that the row is there, and a
  // residual's values the same way: up to 32 waits for memory one after the other, about 10 us a workgroup. 2048 rows, us a
  // launch before and now: the experts' gate/up 157 and 146, their down projection of three super-blocks 126 and 89, a
  // 2048-wide hybrid's mixer inputs on average 131 and 106, 4096 -> 2048 with its residual 56 and 48; 777 rows of 25600 ->
  // 5120 Q6_K 395 and 377, 5120 -> 10240 136 and 118.)
  const uint32_t odd = c & 1u, pairColumn = c - odd;
  constexpr bool kResidual = EP == GGUF_WIDE_RESIDUAL;
  uint32_t residuals[kResidual ? T : 1][2][2];
  if constexpr (kResidual) {
    const uint32_t last = w.rows - 1u;   // (rows past the last read the last)
#pragma unroll
    for (uint32_t t = 0; t < T; ++t)
#pragma unroll
      for (uint32_t r = 0; r < 2; ++r)
#pragma unroll
        for (uint32_t pair = 0; pair < 2; ++pair)
          if (t < tilesHere && w.image[r])
            residuals[t][r][pair] = *reinterpret_cast<const PairBits *>(
                &residual[size_t(min(16u * (tile0 + t) + 4u * kq + 2u * pair + odd, last)) * p.out_stride + column[r] + pairColumn]);
  }
  // a pair's values of the row that this lane stores: its own column's and its neighbour's, in order
  auto trade = [&](float first, float second, float (&out)[2]) __attribute__((always_inline)) {
    const float mine = odd ? second : first, theirs = lane_xor<1>(odd ? first : second);
    out[0] = odd ? theirs : mine;
    out[1] = odd ? mine : theirs;
  };
#pragma unroll
  for (uint32_t t = 0; t < T; ++t) {
    if (t >= tilesHere) break;
    const f32x4 scale = lds.scales[4u * t + kq];
#pragma unroll
    for (uint32_t pair = 0; pair < 2; ++pair) {
      const uint32_t row = 16u * (tile0 + t) + 4u * kq + 2u * pair + odd;
#pragma unroll
      for (uint32_t r = 0; r < (kGateUp ? 1u : 2u); ++r) {
        if (!w.image[r]) continue;
        float value[2], two[2];
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i) {
          const uint32_t v = 2u * pair + i;
          value[i] = acc[r][t][v] * scale[v];
          if constexpr (kGateUp) value[i] = round_bf16(acc[1][t][v] * scale[v]) * silu(round_bf16(value[i]));
        }
        trade(value[0], value[1], two);
        if (row >= w.rows) continue;
        const size_t at = size_t(row) * p.out_stride + column[r] + pairColumn;
        if constexpr (EP == GGUF_WIDE_PARTIAL) {
          *reinterpret_cast<PairFloats *>(static_cast<float *>(out) + size_t(split) * w.rows * p.out_stride + at) = PairFloats{two[0], two[1]};
        } else {
          if constexpr (kResidual) {
            two[0] += bf16_bits_to_float(residuals[t][r][pair] & 0xFFFFu);
            two[1] += bf16_bits_to_float(residuals[t][r][pair] >> 16);
          }
          *reinterpret_cast<PairBits *>(static_cast<uint16_t *>(out) + at) = float_to_bf16_bits(two[0]) | (float_to_bf16_bits(two[1]) << 16);
        }
      }
    }
  }
}
template <uint32_t FMT, uint32_t EP, uint32_t T, bool Staged = false>
__global__ __launch_bounds__(256, 2) void gguf_wide(const uint8_t *__restrict__ seg0, const uint8_t *__restrict__ seg1, const uint8_t *__restrict__ seg2,
                                                    const uint8_t *__restrict__ table, void *__restrict__ out, const uint16_t *__restrict__ residual,
                                                    GgufWideParams p) {
  // The last p.tail_groups column groups are a second part of the grid, in workgroups of four row tiles.
  const uint32_t tallGroups = p.groups - p.tail_groups, tallItems = p.row_groups * p.splits * tallGroups, tallBlocks = (tallItems + 7u) / 8u * 8u;
  const bool tail = T > 4u && blockIdx.x >= tallBlocks;
  const uint32_t block = tail ? blockIdx.x - tallBlocks : blockIdx.x, blocksHere = tail ? gridDim.x - tallBlocks : tallBlocks;
  const uint32_t item = (block % 8u) * (blocksHere / 8u) + block / 8u, rowGroups = tail ? p.tail_row_groups : p.row_groups;
  if (item >= (tail ? p.tail_row_groups * p.tail_groups : tallItems)) return;
  const uint32_t rowGroup = item % rowGroups, rest = item / rowGroups;
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
  const uint32_t blocks = p.input_size / GGUF_BLOCK, liveTiles = (p.rows + 15u) / 16u;
  WideTile w;
  w.split = tail ? 0u : rest % p.splits;
  w.tile0 = liveTiles * rowGroup / rowGroups;
  w.tilesHere = liveTiles * (rowGroup + 1u) / rowGroups - w.tile0;
  w.rows = p.rows;
  w.b0 = blocks * w.split / p.splits;
  w.count = blocks * (w.split + 1u) / p.splits - w.b0;
  wide_columns<FMT, EP == GGUF_WIDE_GATE_UP>(w, seg0, seg1, seg2, p, tail ? tallGroups + rest : rest / p.splits, wave);
  __shared__ uint4 rows0[kWideStageVectors<T>], rows1[kWideStageVectors<T>], rows2[kWideStageVectors<T>], rows3[kWideStageVectors<T>],
      sums[kWideSumVectors<FMT, T, Staged>];
  __shared__ f32x4 scales[kWideScales<T>];
  const WideLds lds{rows0, rows1, rows2, rows3, sums, scales};
  if (tail) wide_workgroup<FMT, EP, 4, Staged>(lds, w, table, out, residual, p);
  else wide_workgroup<FMT, EP, T, Staged>(lds, w, table, out, residual, p);
}
// The routed experts of a prompt chunk: a task is up to T of an expert's row tiles (moe_chunk_place lists them), an item a
// task's column group, the groups of a task side by side. Output rows are the slots'. A workgroup computes whole bodies of
// row tiles, and a tile past the task's multiplies zeros: a kernel of tall tasks holds the bodies of its shorter ones and
// takes the one that fits. A task's weights are converted once, whatever its height: 2048 rows of 128 experts, 8 a row,
// 7 to 10 tiles an expert, in tasks of up to eight 164 and 130 us a layer's gate/up and down, in tasks of five that were
// always computed as five 195 and 151.
template <uint32_t FMT, uint32_t EP, uint32_t T, bool Gathers>
__device__ __forceinline__ void wide_moe(const uint8_t *__restrict__ seg0, const uint8_t *__restrict__ seg1, const uint8_t *__restrict__ table,
                                         void *__restrict__ out, const MoeChunkTask *__restrict__ tasks, const uint32_t *__restrict__ totals,
                                         const uint32_t *__restrict__ slot_row, const GgufWideMoeParams &m) {
  const GgufWideParams &p = m.wide;
  const uint32_t items = totals[1] * p.groups, perDie = (items + 7u) / 8u, item = (blockIdx.x % 8u) * perDie + blockIdx.x / 8u;
  if (blockIdx.x / 8u >= perDie || item >= items) return;
  const MoeChunkTask task = tasks[item / p.groups];
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
  WideTile w;
  w.split = 0;
  w.tile0 = uint32_t(__builtin_amdgcn_readfirstlane(int(task.first_tile)));
  w.tilesHere = uint32_t(__builtin_amdgcn_readfirstlane(int(task.tiles)));
  w.rows = (w.tile0 + w.tilesHere) * 16u;
  w.b0 = 0;
  w.count = p.input_size / GGUF_BLOCK;
  const uint64_t expertAt = task.expert * m.expert_bytes;
  wide_columns<FMT, EP == GGUF_WIDE_GATE_UP>(w, seg0 + expertAt, seg1 + expertAt, seg0 + expertAt, p, item % p.groups, wave);
  __shared__ uint4 rows0[kWideStageVectors<T>], rows1[kWideStageVectors<T>], rows2[kWideStageVectors<T>], rows3[kWideStageVectors<T>],
      sums[kWideSumVectors<FMT, T, false>];
  __shared__ f32x4 scales[kWideScales<T>];
  const WideLds lds{rows0, rows1, rows2, rows3, sums, scales};
  if constexpr (T > 4u) {
    if (w.tilesHere <= 4u) return wide_workgroup<FMT, EP, 4, false, Gathers>(lds, w, table, out, nullptr, p, slot_row);
  }
  if constexpr (T == 8u) {
    if (w.tilesHere == 5u) return wide_workgroup<FMT, EP, 5, false, Gathers>(lds, w, table, out, nullptr, p, slot_row);
    if (w.tilesHere == 6u) return wide_workgroup<FMT, EP, 6, false, Gathers>(lds, w, table, out, nullptr, p, slot_row);
    if (w.tilesHere == 7u) return wide_workgroup<FMT, EP, 7, false, Gathers>(lds, w, table, out, nullptr, p, slot_row);
  }
  wide_workgroup<FMT, EP, T, false, Gathers>(lds, w, table, out, nullptr, p, slot_row);
}
template <uint32_t FMT, uint32_t EP, uint32_t T>
__global__ __launch_bounds__(256, 2) void gguf_wide_moe(const uint8_t *__restrict__ seg0, const uint8_t *__restrict__ seg1, const uint8_t *__restrict__ table,
                                                        void *__restrict__ out, const MoeChunkTask *__restrict__ tasks,
                                                        const uint32_t *__restrict__ totals, GgufWideMoeParams m) {
  wide_moe<FMT, EP, T, false>(seg0, seg1, table, out, tasks, totals, nullptr, m);
}
// The gate/up pair of the rows that the slots gather, from the rows' tables. A table of the slots holds a row as often as it
// has routes, and writing it was a pass bound by memory (16384 slots of 2048 inputs: 27.8 us behind a norm's 9.5, for the 3.8
// that the rows' tables add to the norm's own table). The loads fetch a row's whole lines, as the slots' fetch a tile's, so the
// pair itself takes little longer: 149.3 -> 152.8 us at 2048 rows, 8 of 128 experts, 2048 x 2 x 768 Q4_K.
template <uint32_t FMT, uint32_t T>
__global__ __launch_bounds__(256, 2) void gguf_wide_moe_gathered(const uint8_t *__restrict__ seg0, const uint8_t *__restrict__ seg1,
                                                                 const uint8_t *__restrict__ rows, void *__restrict__ out,
                                                                 const MoeChunkTask *__restrict__ tasks, const uint32_t *__restrict__ totals,
                                                                 const uint32_t *__restrict__ slot_row, GgufWideMoeParams m) {
  wide_moe<FMT, GGUF_WIDE_GATE_UP, T, true>(seg0, seg1, rows, out, tasks, totals, slot_row, m);
}
#define SP_GGUF_WIDE_T(fmt, FMT, T)                                                          \
  SP_REGISTER_KERNEL("gguf_wide_" fmt "_t" #T "_a", (&gguf_wide<FMT, GGUF_WIDE_PLAIN, T>));        \
  SP_REGISTER_KERNEL("gguf_wide_" fmt "_t" #T "_r", (&gguf_wide<FMT, GGUF_WIDE_RESIDUAL, T>));     \
  SP_REGISTER_KERNEL("gguf_wide_" fmt "_t" #T "_g", (&gguf_wide<FMT, GGUF_WIDE_GATE_UP, T>));      \
  SP_REGISTER_KERNEL("gguf_wide_" fmt "_t" #T "_p", (&gguf_wide<FMT, GGUF_WIDE_PARTIAL, T>))
#define SP_GGUF_WIDE(fmt, FMT)  \
  SP_GGUF_WIDE_T(fmt, FMT, 4);  \
  SP_GGUF_WIDE_T(fmt, FMT, 6);  \
  SP_GGUF_WIDE_T(fmt, FMT, 7);  \
  SP_GGUF_WIDE_T(fmt, FMT, 8)
// (the staged rule's chunks are long ones: the tallest tile alone)
#define SP_GGUF_WIDE_STAGED(fmt, FMT)                                                                          \
  SP_REGISTER_KERNEL("gguf_wide_staged_" fmt "_t8_a", (&gguf_wide<FMT, GGUF_WIDE_PLAIN, 8, true>));      \
  SP_REGISTER_KERNEL("gguf_wide_staged_" fmt "_t8_r", (&gguf_wide<FMT, GGUF_WIDE_RESIDUAL, 8, true>));   \
  SP_REGISTER_KERNEL("gguf_wide_staged_" fmt "_t8_g", (&gguf_wide<FMT, GGUF_WIDE_GATE_UP, 8, true>));    \
  SP_REGISTER_KERNEL("gguf_wide_staged_" fmt "_t8_p", (&gguf_wide<FMT, GGUF_WIDE_PARTIAL, 8, true>))
SP_GGUF_WIDE_STAGED("q4k", GGUF_FMT_Q4K);
SP_GGUF_WIDE_STAGED("q5k", GGUF_FMT_Q5K);
SP_GGUF_WIDE_STAGED("q6k", GGUF_FMT_Q6K);
SP_GGUF_WIDE("q4k", GGUF_FMT_Q4K);
SP_GGUF_WIDE("q5k", GGUF_FMT_Q5K);
SP_GGUF_WIDE("q6k", GGUF_FMT_Q6K);

#define SP_GGUF_WIDE_MOE(fmt, FMT, T)                                                             \
  SP_REGISTER_KERNEL("gguf_wide_moe_" fmt "_t" #T "_g", (&gguf_wide_moe<FMT, GGUF_WIDE_GATE_UP, T>)); \
  SP_REGISTER_KERNEL("gguf_wide_moe_" fmt "_t" #T "_x", (&gguf_wide_moe_gathered<FMT, T>)); \
  SP_REGISTER_KERNEL("gguf_wide_moe_" fmt "_t" #T "_a", (&gguf_wide_moe<FMT, GGUF_WIDE_PLAIN, T>))
SP_GGUF_WIDE_MOE("q4k", GGUF_FMT_Q4K, 2);
SP_GGUF_WIDE_MOE("q4k", GGUF_FMT_Q4K, 4);
SP_GGUF_WIDE_MOE("q4k", GGUF_FMT_Q4K, 5);
SP_GGUF_WIDE_MOE("q4k", GGUF_FMT_Q4K, 8);
SP_GGUF_WIDE_MOE("q5k", GGUF_FMT_Q5K, 2);
SP_GGUF_WIDE_MOE("q5k", GGUF_FMT_Q5K, 4);
SP_GGUF_WIDE_MOE("q5k", GGUF_FMT_Q5K, 5);
SP_GGUF_WIDE_MOE("q5k", GGUF_FMT_Q5K, 8);
SP_GGUF_WIDE_MOE("q6k", GGUF_FMT_Q6K, 2);
SP_GGUF_WIDE_MOE("q6k", GGUF_FMT_Q6K, 4);
SP_GGUF_WIDE_MOE("q6k", GGUF_FMT_Q6K, 5);
SP_GGUF_WIDE_MOE("q6k", GGUF_FMT_Q6K, 8);

template <bool Residual, bool Float = false>
__global__ __launch_bounds__(256) void gguf_wide_reduce(const float4 *__restrict__ partials, void *__restrict__ out,
                                                        const uint2 *__restrict__ residual, GgufWideReduceParams p) {
  const uint64_t at = uint64_t(blockIdx.x) * 256u + threadIdx.x, all = uint64_t(p.rows) * (p.columns / 4u);
  if (at >= all) return;
  float4 part[GGUF_WIDE_MAXIMUM_SPLITS];
#pragma unroll
  for (uint32_t s = 0; s < GGUF_WIDE_MAXIMUM_SPLITS; ++s)
    if (s < p.splits) part[s] = partials[s * all + at];
  float4 sum = part[0];
#pragma unroll
  for (uint32_t s = 1; s < GGUF_WIDE_MAXIMUM_SPLITS; ++s)
    if (s < p.splits) sum = make_float4(sum.x + part[s].x, sum.y + part[s].y, sum.z + part[s].z, sum.w + part[s].w);
  if constexpr (Residual) {
    const uint2 r = residual[at];
    sum = make_float4(sum.x + bf16_bits_to_float(r.x & 0xFFFFu), sum.y + bf16_bits_to_float(r.x >> 16), sum.z + bf16_bits_to_float(r.y & 0xFFFFu),
                      sum.w + bf16_bits_to_float(r.y >> 16));
  }
  if constexpr (Float) static_cast<float4 *>(out)[at] = sum;
  else static_cast<uint2 *>(out)[at] = make_uint2(float_to_bf16_bits(sum.x) | (float_to_bf16_bits(sum.y) << 16), float_to_bf16_bits(sum.z) | (float_to_bf16_bits(sum.w) << 16));
}
SP_REGISTER_KERNEL("gguf_wide_reduce_a", &gguf_wide_reduce<false>);
SP_REGISTER_KERNEL("gguf_wide_reduce_f32", (&gguf_wide_reduce<false, true>));
SP_REGISTER_KERNEL("gguf_wide_reduce_r", &gguf_wide_reduce<true>);

} // namespace splash::kernels
