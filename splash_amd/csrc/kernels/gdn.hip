// Gated DeltaNet verify step for gfx950 (the reference's kernels/decode/gdn.metal and
// common/gdn_primitives.h): one workgroup per (value head, lane) runs the short convolution + SiLU,
// the q/k norms and gates of the block's rows, folds the lane's pending (previously accepted) rows
// into the head's 128 x 128 fp32 state, writes THAT state (the one before the block's rows, so a
// rejected row never has to be undone), runs the block's rows for their outputs and gates them.
//
// Sixteen waves. In the prologue and the gate a wave takes a row: lane l holds channels l and 64 + l,
// and a sum over the head's 128 channels is four tree sums over 32 lanes added in channel
// order, the reference's simdgroup sums (gdn.metal:215-222). In the fold a wave advances
// two state rows at once, one per half-wave, lane j of a half holding key columns 4 j .. 4 j + 3;
// the row's products with k are tree sums over the half's 32 lanes, and each token keeps
// the decay, memory, delta, update order of gdn.metal:270-298.
//
// The block's rows never advance the state: every row, of a chain block as of a tree block, takes its
// output from the committed state (the reference does so for tree blocks, gdn.metal:417-478; a chain is
// the tree whose every row follows the row before it): with S_j the state after the j-th token of a
// row's path, S_j z = S_j-1 (d_j (z - c k_j)) + c v_j for c = beta_j (k_j . z), so the row's output is
// S_-1 z_-1 + sum_j c_j v_j; a wave per row walks its path upward for z_-1 and the coefficients, the
// folded state goes to LDS and meets the transformed queries of all rows on the matrix cores, and the
// row's wave adds the path terms before it norms and gates them.
#include "abi/Gdn.h"
#include "abi/Gguf.h"
#include "abi/PagedAttention.h"  // AttentionTreeRow
#include "backend/KernelRegistry.hpp"
#include "kernels/gguf_records.hpp"   // buffer resources
#include "kernels/gguf_wide_table.hpp"

namespace splash::kernels {

namespace {

constexpr uint32_t kDim = GDN_HEAD_DIMENSION, kTaps = GDN_CONVOLUTION_TAPS, kRows = GDN_MAXIMUM_ROWS;
constexpr float kLog2e = 1.44269504089f;

// The sum over each half-wave's 32 lanes (lanes 0..31 and 32..63 apart), in every lane of the half: a
// binary tree over neighbours (pairs, quads, eights, sixteens, the two rows of sixteen), four of its
// levels as row-local DPP operands of the add itself.
template <int Control> __device__ __forceinline__ float dpp_of(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), Control, 0xF, 0xF, false));
}
__device__ __forceinline__ float half_sum(float v) {
  v += dpp_of<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_of<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_of<0x141>(v);  // row_half_mirror: the other quad of the eight
  v += dpp_of<0x140>(v);  // row_mirror: the other eight of the row
  v += __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, v), 0x401F));  // lane ^ 16
  return v;
}
// The sum of a head's 128 values, lane l holding a = value[l] and b = value[64 + l]: the four
// 32-channel groups' sums added in channel order.
__device__ __forceinline__ float head_sum(float a, float b) {
  const float first = half_sum(a), second = half_sum(b);
  const float s0 = lane_value_of(first, 0), s1 = lane_value_of(first, 32), s2 = lane_value_of(second, 0), s3 = lane_value_of(second, 32);
  return ((s0 + s1) + s2) + s3;
}
__device__ __forceinline__ uint32_t path_row(uint32_t path, uint32_t depth) {
  for (uint32_t i = 0; i < depth; ++i) path &= path - 1u;
  return uint32_t(__builtin_ctz(path));
}
__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float silu_of(float x) { return x / (1.0f + exp2_fast(-kLog2e * x)); }
__device__ __forceinline__ float sigmoid_of(float x) { return 1.0f / (1.0f + exp2_fast(-kLog2e * x)); }

struct Tape {
  uint16_t *inputs, *kv;
  float *decay;
  uint16_t *beta;
};
__device__ __forceinline__ Tape tape_at(uint8_t *tape, uint64_t offset, const GdnShapeParams &s) {
  const uint32_t kvWidth = (s.key_heads + s.value_heads) * kDim;
  uint8_t *layer = tape + offset;
  return {reinterpret_cast<uint16_t *>(layer), reinterpret_cast<uint16_t *>(layer + gdn_tape_kv_offset(s.conv_dim)),
          reinterpret_cast<float *>(layer + gdn_tape_decay_offset(s.conv_dim, kvWidth)),
          reinterpret_cast<uint16_t *>(layer + gdn_tape_beta_offset(s.conv_dim, kvWidth, s.value_heads))};
}

// The rows a head folds into its state: k, v and gates, in LDS.
struct Pending {
  uint16_t keys[kRows][kDim];
  uint16_t values[kRows][kDim];
  float decay[kRows];
  uint16_t beta[kRows];
};

// Path row `row` of a tape to slot `slot`: one wave, lane l the channels l and 64 + l.
__device__ __forceinline__ void load_pending(const Tape &tape, Pending &pending, uint32_t slot, uint32_t row, uint32_t head,
                                             const GdnShapeParams &s, uint32_t lane) {
  const uint32_t keyWidth = s.key_heads * kDim, kvWidth = keyWidth + s.value_heads * kDim;
  const uint32_t keyHead = head / (s.value_heads / s.key_heads);
  const uint16_t *source = tape.kv + size_t(row) * kvWidth;
#pragma unroll
  for (uint32_t part = 0; part < 2; ++part) {
    const uint32_t d = lane + 64u * part;
    pending.keys[slot][d] = source[keyHead * kDim + d];
    pending.values[slot][d] = source[keyWidth + head * kDim + d];
  }
  if (lane == 0) {
    pending.decay[slot] = tape.decay[row * s.value_heads + head];
    pending.beta[slot] = tape.beta[row * s.value_heads + head];
  }
}

// The three rows of convolution inputs before a command's first row, after `consumed` rows of
// `path` of `rows` (gdn_primitives.h:20-35).
struct History {
  const uint16_t *row[kTaps - 1];
  // Row `index` by selects: an indexed read would keep the rows in scratch.
  __device__ __forceinline__ const uint16_t *at(uint32_t index) const { return index == 0 ? row[0] : index == 1 ? row[1] : row[2]; }
};
__device__ __forceinline__ History history_of(const uint16_t *carried, const uint16_t *rows, uint32_t conv_dim, uint32_t consumed,
                                              uint32_t path) {
  History h;
#pragma unroll
  for (uint32_t r = 0; r < kTaps - 1; ++r) {
    const uint32_t source = consumed + r;
    h.row[r] = source < kTaps - 1 ? carried + size_t(source) * conv_dim : rows + size_t(path_row(path, source - (kTaps - 1))) * conv_dim;
  }
  return h;
}

// A row's convolution + SiLU of one channel from its four taps, oldest first (gdn_primitives.h:37-50).
__device__ __forceinline__ float conv_silu(const uint16_t *const (&taps)[kTaps], const uint16_t *conv_weights, uint32_t channel) {
  float value = 0.f;
#pragma unroll
  for (uint32_t tap = 0; tap < kTaps; ++tap)
    value += bf16_bits_to_float(taps[tap][channel]) * bf16_bits_to_float(conv_weights[size_t(channel) * kTaps + tap]);
  value = round_bf16(value);
  return round_bf16(silu_of(value));
}

// A row's normalized, scaled query and key and its value of one head as bf16 bits, lane l the
// dimensions l and 64 + l (gdn.metal:198-232): q and k are RMS-normed over the head, rounded, then
// scaled by 1/128 and 1/sqrt(128).
struct HeadRow {
  uint32_t query[2], key[2], value[2];
};
__device__ __forceinline__ HeadRow head_row(const uint16_t *const (&taps)[kTaps], const uint16_t *conv_weights, uint32_t qChannel,
                                            uint32_t kChannel, uint32_t vChannel, uint32_t lane) {
  float q[2], k[2], v[2];
#pragma unroll
  for (uint32_t part = 0; part < 2; ++part) {
    const uint32_t d = lane + 64u * part;
    q[part] = conv_silu(taps, conv_weights, qChannel + d);
    k[part] = conv_silu(taps, conv_weights, kChannel + d);
    v[part] = conv_silu(taps, conv_weights, vChannel + d);
  }
  const float qScale = 1.0f / sqrtf(head_sum(q[0] * q[0], q[1] * q[1]) / float(kDim) + 1e-6f);
  const float kScale = 1.0f / sqrtf(head_sum(k[0] * k[0], k[1] * k[1]) / float(kDim) + 1e-6f);
  HeadRow row;
#pragma unroll
  for (uint32_t part = 0; part < 2; ++part) {
    row.query[part] = float_to_bf16_bits(round_bf16(q[part] * qScale) * 0.0078125f);
    row.key[part] = float_to_bf16_bits(round_bf16(k[part] * kScale) * 0.08838834765f);
    row.value[part] = float_to_bf16_bits(v[part]);
  }
  return row;
}

// A row's gates of one value head (gdn_primitives.h:65-73): beta = bf16(sigmoid(b)); decay =
// exp(a_scale bf16(softplus(bf16(a + dt_bias)))).
struct Gates {
  uint32_t beta;
  float decay;
};
__device__ __forceinline__ Gates gates_of(const uint16_t *inputs, uint32_t bOffset, uint32_t aOffset, uint32_t head,
                                          const float *a_scale, const uint16_t *dt_bias) {
  Gates g;
  g.beta = float_to_bf16_bits(sigmoid_of(bf16_bits_to_float(inputs[bOffset + head])));
  const float x = round_bf16(bf16_bits_to_float(inputs[aOffset + head]) + bf16_bits_to_float(dt_bias[head]));
  const float softplus = round_bf16(fmaxf(x, 0.0f) + __builtin_amdgcn_logf(1.0f + exp2_fast(-kLog2e * fabsf(x))) * 0.69314718056f);
  g.decay = exp2_fast(kLog2e * (a_scale[head] * softplus));
  return g;
}

// The gated output norm of a row's 128 recurrent values of one head, lane l the dimensions l and
// 64 + l, as bf16 bits (gdn.metal:489-526): RMS norm with the mixer's weight, rounded, times silu(z)
// (or sigmoid(z)) of the row's gate columns `z`.
__device__ __forceinline__ float norm_weight_of(const void *norm_weight, uint32_t flags, uint32_t d) {
  return (flags & GDN_FLOAT_NORM) ? static_cast<const float *>(norm_weight)[d] : bf16_bits_to_float(static_cast<const uint16_t *>(norm_weight)[d]);
}
__device__ __forceinline__ void gated_values(const float (&value)[2], const float (&weight)[2], const float (&z)[2], uint32_t flags,
                                             uint32_t (&bits)[2]) {
  const float inverse = 1.0f / sqrtf(head_sum(value[0] * value[0], value[1] * value[1]) / float(kDim) + 1e-6f);
#pragma unroll
  for (uint32_t part = 0; part < 2; ++part) {
    const float normalized = round_bf16((value[part] * inverse) * weight[part]);
    const float gated = (normalized * ((flags & GDN_SIGMOID_GATE) ? 1.0f : z[part])) / (1.0f + exp2_fast(-kLog2e * z[part]));
    bits[part] = float_to_bf16_bits(gated);
  }
}
__device__ __forceinline__ void gated_norm(const float (&value)[2], const void *norm_weight, uint32_t flags, const uint16_t *z_row,
                                           uint32_t lane, uint32_t (&bits)[2]) {
  float weight[2], z[2];
#pragma unroll
  for (uint32_t part = 0; part < 2; ++part) {
    weight[part] = norm_weight_of(norm_weight, flags, lane + 64u * part);
    z[part] = bf16_bits_to_float(z_row[lane + 64u * part]);
  }
  gated_values(value, weight, z, flags, bits);
}

// One token's delta-rule step on the wave's state rows (R pairs, a row per half-wave): decay,
// memory, delta, update (gdn.metal:270-298). k: the lane's four key columns; value: each row's value.
template <int R>
__device__ __forceinline__ void advance_rows(float (&state)[R][4], const float (&k)[4], const float (&value)[R], float decay, float beta) {
  float memory[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    memory[r] = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      state[r][i] *= decay;
      memory[r] += state[r][i] * k[i];
    }
    memory[r] = half_sum(memory[r]);
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float delta = (value[r] - memory[r]) * beta;
#pragma unroll
    for (int i = 0; i < 4; ++i) state[r][i] += k[i] * delta;
  }
}
// The same from a token's staged key row and value row (bf16 in LDS).
template <int R>
__device__ __forceinline__ void advance(float (&state)[R][4], const uint16_t *key, const uint16_t *value_row, const uint32_t (&value_dim)[R],
                                        float decay, float beta, uint32_t column) {
  const uint2 kb = *reinterpret_cast<const uint2 *>(key + column);
  const float k[4] = {bf16_bits_to_float(kb.x & 0xFFFFu), bf16_bits_to_float(kb.x >> 16), bf16_bits_to_float(kb.y & 0xFFFFu),
                      bf16_bits_to_float(kb.y >> 16)};
  float value[R];
#pragma unroll
  for (int r = 0; r < R; ++r) value[r] = bf16_bits_to_float(value_row[value_dim[r]]);
  advance_rows<R>(state, k, value, decay, beta);
}

constexpr int kInFlight = 4;  // row pairs a wave advances together, to overlap their reductions
constexpr uint32_t kWaves = 16;  // of a workgroup: with four pairs each they hold the head's 128 state rows at once

} // namespace

// gdn_decode: grid (value_heads, lanes), 1024 threads. `tree` holds the step's rows' places in their
// blocks (bit j of a row's ancestors: row j of its block is on its path, itself included).
__global__ __launch_bounds__(64 * kWaves) void gdn_decode(const uint16_t *__restrict__ packed, const uint16_t *__restrict__ conv_weights,
                                                  uint8_t *__restrict__ states, uint8_t *__restrict__ tape,
                                                  const float *__restrict__ a_scale, const uint16_t *__restrict__ dt_bias,
                                                  const void *__restrict__ norm_weight, uint16_t *__restrict__ hidden,
                                                  const AttentionTreeRow *__restrict__ tree, uint8_t *__restrict__ table,
                                                  GdnDecodeParams p) {
  __shared__ __align__(16) uint16_t queries[kRows][kDim], keys[kRows][kDim], values[kRows][kDim], outputs[kRows][kDim];
  __shared__ __align__(16) float transformed[kRows][kDim + 4], committed[kDim][kDim + 4];   // rows of sixteen lanes in sixteen bank groups
  __shared__ float products[2][kRows][kDim + 4], coefficients[kRows][kRows];
  __shared__ float decays[kRows];
  __shared__ uint16_t betas[kRows];
  __shared__ uint32_t paths[kRows];
  __shared__ __align__(16) Pending pending;

  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, head = blockIdx.x;
  const GdnShapeParams s = p.shape;
  const GdnLane L = p.lane[blockIdx.y];
  const uint32_t perKey = s.value_heads / s.key_heads, keyHead = head / perKey, keyWidth = s.key_heads * kDim;
  const uint32_t kvWidth = keyWidth + s.value_heads * kDim, C = s.conv_dim, P = s.packed_width;
  const uint32_t zOffset = C, bOffset = C + s.value_heads * kDim, aOffset = bOffset + s.value_heads;
  const bool sharedWriter = head % perKey == 0;
  const uint32_t rows = L.rows, pendingRows = uint32_t(__builtin_popcount(L.pending_path));
  const uint16_t *rowsIn = packed + size_t(L.first_row) * P;

  const uint8_t *current = states + L.current_cell;
  uint8_t *next = states + L.next_cell;
  const uint16_t *convIn = reinterpret_cast<const uint16_t *>(current + uint64_t(p.layer) * p.conv_layer_bytes);
  uint16_t *convOut = reinterpret_cast<uint16_t *>(next + uint64_t(p.layer) * p.conv_layer_bytes);
  const float *stateIn = reinterpret_cast<const float *>(current + p.convolution_state_bytes + uint64_t(p.layer) * p.recurrent_layer_bytes);
  float *stateOut = reinterpret_cast<float *>(next + p.convolution_state_bytes + uint64_t(p.layer) * p.recurrent_layer_bytes);
  const Tape pendingTape = tape_at(tape, L.pending_tape, s), stepTape = tape_at(tape, L.step_tape, s);
  const History history = history_of(convIn, pendingTape.inputs, C, pendingRows, L.pending_path);

  // ---- prologue ----
  // channels of this head: q and k of its key head, its v; lane l the dimensions l and 64 + l
  const uint32_t qChannel = keyHead * kDim, kChannel = keyWidth + keyHead * kDim, vChannel = 2 * keyWidth + head * kDim;
  // The state's carried rows after the pending path: waves 0..2 hold one each until the block's rows are done.
  uint16_t carryV[2] = {0, 0}, carryQ[2] = {0, 0}, carryK[2] = {0, 0};
  if (wave < kTaps - 1) {
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part) {
      const uint32_t d = lane + 64u * part;
      carryV[part] = history.at(wave)[vChannel + d];
      if (sharedWriter) {
        carryQ[part] = history.at(wave)[qChannel + d];
        carryK[part] = history.at(wave)[kChannel + d];
      }
    }
  }
  for (uint32_t token = wave; token < pendingRows; token += kWaves)
    load_pending(pendingTape, pending, token, path_row(L.pending_path, token), head, s, lane);
  for (uint32_t token = wave; token < rows; token += kWaves) {
    // The row's path within the block (its own row the last), its depth, and the block rows of its
    // last four path tokens; taps before the block's first row read the history (gdn.metal:198-206).
    const uint32_t path = (tree[L.first_row + token].ancestors & ((1u << token) - 1u)) | (1u << token);
    const uint32_t depth = uint32_t(__builtin_popcount(path)) - 1u;
    const uint16_t *taps[kTaps];
    {
      uint32_t up = path;
#pragma unroll
      for (uint32_t tap = kTaps; tap-- > 0;) {
        const uint32_t row = up ? 31u - uint32_t(__builtin_clz(up)) : 0u;
        up &= ~(1u << row);
        taps[tap] = depth + tap < kTaps - 1 ? history.at(depth + tap) : rowsIn + size_t(row) * P;
      }
    }
    const HeadRow row = head_row(taps, conv_weights, qChannel, kChannel, vChannel, lane);
    const uint16_t *inputs = rowsIn + size_t(token) * P;
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part) {
      const uint32_t d = lane + 64u * part;
      queries[token][d] = uint16_t(row.query[part]);
      keys[token][d] = uint16_t(row.key[part]);
      values[token][d] = uint16_t(row.value[part]);
      stepTape.inputs[size_t(token) * C + vChannel + d] = inputs[vChannel + d];
      stepTape.kv[size_t(token) * kvWidth + keyWidth + head * kDim + d] = uint16_t(row.value[part]);
      if (sharedWriter) {
        stepTape.inputs[size_t(token) * C + qChannel + d] = inputs[qChannel + d];
        stepTape.inputs[size_t(token) * C + kChannel + d] = inputs[kChannel + d];
        stepTape.kv[size_t(token) * kvWidth + keyHead * kDim + d] = uint16_t(row.key[part]);
      }
    }
    if (lane == 0) {
      const Gates gates = gates_of(inputs, bOffset, aOffset, head, a_scale, dt_bias);
      stepTape.beta[token * s.value_heads + head] = uint16_t(gates.beta);
      stepTape.decay[token * s.value_heads + head] = gates.decay;
      betas[token] = uint16_t(gates.beta);
      decays[token] = gates.decay;
      paths[token] = path;
    }
  }
  if (wave < kTaps - 1) {
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part) {
      const uint32_t d = lane + 64u * part;
      convOut[size_t(wave) * C + vChannel + d] = carryV[part];
      if (sharedWriter) {
        convOut[size_t(wave) * C + qChannel + d] = carryQ[part];
        convOut[size_t(wave) * C + kChannel + d] = carryK[part];
      }
    }
  }
  __syncthreads();

  {
    // ---- tree rows: transformed queries and path coefficients, a wave per row ----
    const uint32_t j = lane & 31u, column = 4u * j;
    for (uint32_t token = wave; token < rows; token += kWaves) {
      const uint2 qb = *reinterpret_cast<const uint2 *>(&queries[token][column]);
      float z[4] = {bf16_bits_to_float(qb.x & 0xFFFFu), bf16_bits_to_float(qb.x >> 16), bf16_bits_to_float(qb.y & 0xFFFFu),
                    bf16_bits_to_float(qb.y >> 16)};
      float coefficient = 0.f;
      for (uint32_t up = paths[token]; up;) {
        const uint32_t row = 31u - uint32_t(__builtin_clz(up));
        up &= ~(1u << row);
        const uint2 kb = *reinterpret_cast<const uint2 *>(&keys[row][column]);
        const float k[4] = {bf16_bits_to_float(kb.x & 0xFFFFu), bf16_bits_to_float(kb.x >> 16), bf16_bits_to_float(kb.y & 0xFFFFu),
                            bf16_bits_to_float(kb.y >> 16)};
        float product = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) product += k[i] * z[i];
        const float c = bf16_bits_to_float(betas[row]) * half_sum(product);
        const float d = decays[row];
#pragma unroll
        for (int i = 0; i < 4; ++i) z[i] = d * (z[i] - c * k[i]);
        if (j == row) coefficient = c;
      }
      if (lane < 32u) {
        *reinterpret_cast<float4 *>(&transformed[token][column]) = make_float4(z[0], z[1], z[2], z[3]);
        if (j < kRows) coefficients[token][j] = coefficient;
      }
    }
    __syncthreads();
  }

  // ---- recurrence ----
  {
    const uint32_t half = lane >> 5, column = 4u * (lane & 31u);
    for (uint32_t batch = 0; batch < kDim / (2u * kWaves); batch += kInFlight) {
      uint32_t valueDim[kInFlight];
      float state[kInFlight][4];
#pragma unroll
      for (int r = 0; r < kInFlight; ++r) {
        valueDim[r] = (batch + r) * 2u * kWaves + wave * 2u + half;
        const float4 loaded = *reinterpret_cast<const float4 *>(stateIn + (size_t(head) * kDim + valueDim[r]) * kDim + column);
        state[r][0] = loaded.x;
        state[r][1] = loaded.y;
        state[r][2] = loaded.z;
        state[r][3] = loaded.w;
      }
      for (uint32_t token = 0; token < pendingRows; ++token)
        advance<kInFlight>(state, pending.keys[token], pending.values[token], valueDim, pending.decay[token],
                           bf16_bits_to_float(pending.beta[token]), column);
#pragma unroll
      for (int r = 0; r < kInFlight; ++r)
        *reinterpret_cast<float4 *>(stateOut + (size_t(head) * kDim + valueDim[r]) * kDim + column) =
            make_float4(state[r][0], state[r][1], state[r][2], state[r][3]);
#pragma unroll
      for (int r = 0; r < kInFlight; ++r)
        *reinterpret_cast<float4 *>(&committed[valueDim[r]][column]) = make_float4(state[r][0], state[r][1], state[r][2], state[r][3]);
    }
  }
  __syncthreads();

  // ---- the committed state's products with the transformed queries (gdn.metal:363-377): wave w sixteen of the state's
  // rows over half of their columns, for all the block's tokens (a token past them is a product that nothing reads). One
  // matrix instruction's sums of four products each, added as a tree: against 64 bits 6.2e-8 of the terms' norm where a
  // half-wave's tree of four-term chains is off by 6.6e-8 (tests/test_gdn_products_gpu.py). A block's rows were 0.8 us each
  // in the state's registers, four 32-lane sums a wave; the kernel at 32 heads, as many pending rows as rows: 8 lanes of 16
  // rows 42.0 -> 32.8 us, of 4 19.2 -> 17.5, of 1 13.3 -> 13.7 (one form for every count, so that a row's bits do not depend
  // on its block's). ----
  {
    const uint32_t tile = wave >> 1, from = (kDim / 2u) * (wave & 1u), line = lane & 15u, quarter = lane >> 4;
    const f32x4 none = {};
    f32x4 sums[4];
#pragma unroll
    for (uint32_t c = 0; c < 4; ++c) {
      const float4 z = *reinterpret_cast<const float4 *>(&transformed[line][from + 16u * c + 4u * quarter]);
      const float4 m = *reinterpret_cast<const float4 *>(&committed[16u * tile + line][from + 16u * c + 4u * quarter]);
      sums[c] = (__builtin_amdgcn_mfma_f32_16x16x4f32(z.x, m.x, none, 0, 0, 0) + __builtin_amdgcn_mfma_f32_16x16x4f32(z.y, m.y, none, 0, 0, 0)) +
                (__builtin_amdgcn_mfma_f32_16x16x4f32(z.z, m.z, none, 0, 0, 0) + __builtin_amdgcn_mfma_f32_16x16x4f32(z.w, m.w, none, 0, 0, 0));
    }
    const f32x4 sum = (sums[0] + sums[1]) + (sums[2] + sums[3]);
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) products[wave & 1u][4u * quarter + i][16u * tile + line] = sum[i];
  }
  __syncthreads();

  // ---- gated output norm (gdn.metal:489-526) ----
  const uint32_t outHead = (p.flags & GDN_TILED_HEADS) ? (head % perKey) * s.key_heads + head / perKey : head;
  for (uint32_t token = wave; token < rows; token += kWaves) {
    // beside the products the path's terms, in block order: rows off the path are not touched, whatever they hold
    float value[2] = {0.f, 0.f};
    for (uint32_t path = paths[token]; path; path &= path - 1u) {
      const uint32_t row = uint32_t(__builtin_ctz(path));
#pragma unroll
      for (uint32_t part = 0; part < 2; ++part)
        value[part] = __fmaf_rn(coefficients[token][row], bf16_bits_to_float(values[row][lane + 64u * part]), value[part]);
    }
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part)
      value[part] = round_bf16(value[part] + (products[0][token][lane + 64u * part] + products[1][token][lane + 64u * part]));
    uint32_t gated[2];
    gated_norm(value, norm_weight, p.flags, rowsIn + size_t(token) * P + zOffset + head * kDim, lane, gated);
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part) {
      const uint32_t d = lane + 64u * part;
      hidden[(size_t(L.first_row + token) * s.value_heads + outHead) * kDim + d] = uint16_t(gated[part]);
      outputs[token][d] = uint16_t(gated[part]);  // this wave's row: read above, and below for the table
    }
    if (p.table_tiles) {
      // The row's 128 values of this head as 32 runs of four inputs, a lane a run: the pieces, and the sums of 16
      // and 32 inputs in input order, that gguf_prepare_table would write of the hidden rows.
      const uint32_t packedRow = L.first_row + token, r = packedRow % 16u, width = s.value_heads * kDim, G = width / 32u;
      const uint32_t piece = packedRow / 16u / GGUF_PIECE_TILES, tile = packedRow / 16u % GGUF_PIECE_TILES;
      const uint32_t tiles = min(uint32_t(GGUF_PIECE_TILES), p.table_tiles - piece * GGUF_PIECE_TILES);
      uint8_t *mine = table + piece * gguf_table_bytes(width, GGUF_PIECE_TILES);
      const uint32_t run = lane & 31u, q = outHead * (kDim / 4u) + run, g = q / 8u, half = (q / 4u) % 2u, kq = q % 4u;
      const uint2 raw = *reinterpret_cast<const uint2 *>(&outputs[token][4u * run]);
      const uint32_t x0 = raw.x & 0xFFFFu, x1 = raw.x >> 16, x2 = raw.y & 0xFFFFu, x3 = raw.y >> 16;
      float sum = (bf16_bits_to_float(x0) + bf16_bits_to_float(x1)) + (bf16_bits_to_float(x2) + bf16_bits_to_float(x3));
      const float s1 = lane_down<1>(sum), s2 = lane_down<2>(sum), s3 = lane_down<3>(sum);
      sum = ((sum + s1) + s2) + s3;
      const float other = lane_down<4>(sum);
      if (lane < 32u) {
        // operand elements 4 half + {0,1,2,3} are inputs 4 kq + {0,2,1,3} of the half
        reinterpret_cast<uint2 *>(mine)[((size_t(tile) * G + g) * 64u + kq * 16u + r) * 2u + half] = make_uint2(x0 | (x2 << 16), x1 | (x3 << 16));
        if (kq == 0) {
          float *sums32 = reinterpret_cast<float *>(mine + gguf_table_sums32_offset(width, tiles));
          float *sums16 = reinterpret_cast<float *>(mine + gguf_table_sums16_offset(width, tiles));
          sums16[(size_t(tile) * 2u * G + 2u * g + half) * 16u + r] = sum;
          if (half == 0) sums32[(size_t(tile) * G + g) * 16u + r] = sum + other;
        }
      }
    }
  }
}
SP_REGISTER_KERNEL("gdn_decode", &gdn_decode);

// gdn_fold: grid (value_heads, layers), 1024 threads (gdn.metal:630-698, exact cells).
__global__ __launch_bounds__(64 * kWaves) void gdn_fold(uint8_t *__restrict__ states, uint8_t *__restrict__ tape,
                                                const uint32_t *__restrict__ retained, GdnFoldParams p) {
  __shared__ __align__(16) Pending pending;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, head = blockIdx.x, layer = blockIdx.y;
  const GdnShapeParams s = p.shape;
  const uint32_t rows = p.rows, path = retained[0];
  if (uint32_t(__builtin_popcount(path)) < rows) return;
  const uint32_t perKey = s.value_heads / s.key_heads, keyHead = head / perKey, keyWidth = s.key_heads * kDim, C = s.conv_dim;
  const Tape step = tape_at(tape, p.step_tape + uint64_t(layer) * p.tape_layer_bytes, s);
  const uint8_t *cell = states + p.state_cell;
  uint8_t *fold = states + p.fold_cell;
  for (uint32_t token = wave; token < rows; token += kWaves) load_pending(step, pending, token, path_row(path, token), head, s, lane);
  if (wave < kTaps - 1) {
    const History history = history_of(reinterpret_cast<const uint16_t *>(cell + uint64_t(layer) * p.conv_layer_bytes), step.inputs, C, rows, path);
    uint16_t *carried = reinterpret_cast<uint16_t *>(fold + uint64_t(layer) * p.conv_layer_bytes) + size_t(wave) * C;
    const uint32_t qChannel = keyHead * kDim, kChannel = keyWidth + keyHead * kDim, vChannel = 2 * keyWidth + head * kDim;
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part) {
      const uint32_t d = lane + 64u * part;
      carried[vChannel + d] = history.row[wave][vChannel + d];
      if (head % perKey == 0) {
        carried[qChannel + d] = history.row[wave][qChannel + d];
        carried[kChannel + d] = history.row[wave][kChannel + d];
      }
    }
  }
  __syncthreads();
  const float *stateIn = reinterpret_cast<const float *>(cell + p.convolution_state_bytes + uint64_t(layer) * p.recurrent_layer_bytes);
  float *stateOut = reinterpret_cast<float *>(fold + p.convolution_state_bytes + uint64_t(layer) * p.recurrent_layer_bytes);
  const uint32_t half = lane >> 5, column = 4u * (lane & 31u);
  for (uint32_t batch = 0; batch < kDim / (2u * kWaves); batch += kInFlight) {
    uint32_t valueDim[kInFlight];
    float state[kInFlight][4];
#pragma unroll
    for (int r = 0; r < kInFlight; ++r) {
      valueDim[r] = (batch + r) * 2u * kWaves + wave * 2u + half;
      const float4 loaded = *reinterpret_cast<const float4 *>(stateIn + (size_t(head) * kDim + valueDim[r]) * kDim + column);
      state[r][0] = loaded.x;
      state[r][1] = loaded.y;
      state[r][2] = loaded.z;
      state[r][3] = loaded.w;
    }
    for (uint32_t token = 0; token < rows; ++token)
      advance<kInFlight>(state, pending.keys[token], pending.values[token], valueDim, pending.decay[token],
                         bf16_bits_to_float(pending.beta[token]), column);
#pragma unroll
    for (int r = 0; r < kInFlight; ++r)
      *reinterpret_cast<float4 *>(stateOut + (size_t(head) * kDim + valueDim[r]) * kDim + column) =
          make_float4(state[r][0], state[r][1], state[r][2], state[r][3]);
  }
}
SP_REGISTER_KERNEL("gdn_fold", &gdn_fold);

// ---- prefill: a prompt chunk, whose rows all enter the state (the reference's kernels/prefill/gdn.metal) ----
//
// Three passes over a run of `tokens` rows of one lane and layer. The rows' k, v and gates are those
// a verify step would leave on its tape for the same rows (the same device functions compute both) and
// a state row's recurrence is `advance`, the fold's: a prompt that enters the state through these
// kernels leaves the cell, bit for bit, that the same rows leave when they enter as accepted verify
// blocks. Only the outputs differ in form: here a row reads the state after its own token, o = S_t q_t
// (gdn.metal:291-298), where a verify block's rows read the state before the block.

// gdn_prefill_prepare: grid (2 key_heads + value_heads, ceil(tokens / (4 GDN_PREPARE_ROWS))), 256 threads, a wave per run
// of GDN_PREPARE_ROWS rows and head of the convolution's channels (the query heads, the key heads, then the value heads),
// lane l the dimensions l and 64 + l: convolution + SiLU, the norm of a query or key head, a value head's gates with a
// lane a row (prefill/gdn.metal:196-262). The workgroups of the first rows also write the convolution carry after the
// run's last row. Bound by its vector instructions (silu's correctly rounded division, the roundings): a wave reads a
// row's inputs and widens them once for the four taps that use them, and a key head that two value heads share is worked
// out once, where a wave per (row, value head) did both over again. 2048 rows of 16 / 32 heads: 63 us that way, 34 so.
__global__ __launch_bounds__(256) void gdn_prefill_prepare(const uint16_t *__restrict__ packed, const uint16_t *__restrict__ conv_weights,
                                                           uint8_t *__restrict__ states, const float *__restrict__ a_scale,
                                                           const uint16_t *__restrict__ dt_bias, uint16_t *__restrict__ queries,
                                                           uint16_t *__restrict__ keys, uint16_t *__restrict__ values,
                                                           float *__restrict__ decay, uint16_t *__restrict__ beta, GdnPrefillParams p) {
  constexpr uint32_t R = GDN_PREPARE_ROWS;
  const uint32_t lane = threadIdx.x & 63u, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6))), unit = blockIdx.x;
  const uint32_t firstRow = (blockIdx.y * 4u + wave) * R;
  const GdnShapeParams s = p.shape;
  const uint32_t keyWidth = s.key_heads * kDim, valueWidth = s.value_heads * kDim, C = s.conv_dim, P = s.packed_width;
  const uint32_t bOffset = C + valueWidth, aOffset = bOffset + s.value_heads, channel = unit * kDim;
  const uint16_t *convIn = reinterpret_cast<const uint16_t *>(states + p.current_cell + uint64_t(p.layer) * p.conv_layer_bytes);
  uint16_t *convOut = reinterpret_cast<uint16_t *>(states + p.next_cell + uint64_t(p.layer) * p.conv_layer_bytes);
  // input position i of the run's history: the carried rows, then the run's own (gdn_primitives.h:20-35)
  auto input = [&](uint32_t position) __attribute__((always_inline)) -> const uint16_t * {
    return position < kTaps - 1 ? convIn + size_t(position) * C : packed + size_t(p.first + position - (kTaps - 1)) * P;
  };
  if (blockIdx.y == 0 && wave < kTaps - 1) {
    const uint16_t *source = input(p.tokens + wave);
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part) convOut[size_t(wave) * C + channel + lane + 64u * part] = source[channel + lane + 64u * part];
  }
  if (firstRow >= p.tokens) return;
  const uint32_t rows = min(R, p.tokens - firstRow);
  float taps[2][kTaps], inputs[2][R + kTaps - 1];
#pragma unroll
  for (uint32_t part = 0; part < 2; ++part) {
    const uint32_t d = channel + lane + 64u * part;
#pragma unroll
    for (uint32_t i = 0; i < R + kTaps - 1; ++i)   // the last row's last input again past the run's end
      inputs[part][i] = bf16_bits_to_float(input(firstRow + min(i, rows + kTaps - 2u))[d]);
#pragma unroll
    for (uint32_t tap = 0; tap < kTaps; ++tap) taps[part][tap] = bf16_bits_to_float(conv_weights[size_t(d) * kTaps + tap]);
  }
  const size_t at = size_t(p.first) + firstRow;  // the run of rows' place in the chunk's buffers
  const bool query = unit < s.key_heads, key = !query && unit < 2u * s.key_heads;
  uint16_t *out = (query ? queries + at * keyWidth + channel : key ? keys + at * keyWidth + (channel - keyWidth)
                                                                  : values + at * valueWidth + (channel - 2u * keyWidth)) + lane;
  const uint32_t width = query || key ? keyWidth : valueWidth;
  const float scaleAfter = query ? 0.0078125f : 0.08838834765f;
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    if (r >= rows) break;
    float x[2];
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part) {
      float value = 0.f;   // conv_silu's sum
#pragma unroll
      for (uint32_t tap = 0; tap < kTaps; ++tap) value += inputs[part][r + tap] * taps[part][tap];
      x[part] = round_bf16(silu_of(round_bf16(value)));
    }
    if (query || key) {
      const float scale = 1.0f / sqrtf(head_sum(x[0] * x[0], x[1] * x[1]) / float(kDim) + 1e-6f);
#pragma unroll
      for (uint32_t part = 0; part < 2; ++part) x[part] = round_bf16(x[part] * scale) * scaleAfter;
    }
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part) out[size_t(r) * width + 64u * part] = uint16_t(float_to_bf16_bits(x[part]));
  }
  if (!query && !key && lane < rows) {
    const uint32_t head = unit - 2u * s.key_heads;
    const size_t row = at + lane;
    const Gates gates = gates_of(packed + row * P, bOffset, aOffset, head, a_scale, dt_bias);
    beta[row * s.value_heads + head] = uint16_t(gates.beta);
    decay[row * s.value_heads + head] = gates.decay;
  }
}
SP_REGISTER_KERNEL("gdn_prefill_prepare", &gdn_prefill_prepare);

// gdn_prefill_scan: grid (value_heads * 128 / GDN_SCAN_STATE_ROWS), 256 threads. A workgroup carries GDN_SCAN_STATE_ROWS
// rows of a head's state through the run in registers, token by token (prefill/gdn.metal:11-23): a wave holds four rows,
// a row per sixteen lanes, lane j of them the key columns 8 j .. 8 j + 7. A row's sums over the columns are the fold's tree:
// its lanes of four columns pair up inside a lane here, and the four levels left are row-local DPP adds, where a row over
// 32 lanes ends with a trip through the LDS pipe. The pass is bound by the instructions of a token's dependent chain: four
// rows a wave for the instructions that two took (keys and queries are widened once, when they are staged). 2048 tokens
// of 32 heads: 715 -> 400 us.
// Blocks of GDN_SCAN_BLOCK tokens of k, q, v and gates are staged in LDS while the block after them is in flight to
// registers; a block's outputs collect in LDS and leave as whole 16-byte runs.
__device__ __forceinline__ float sixteen_sum(float v) {
  v += dpp_of<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_of<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_of<0x141>(v);  // row_half_mirror
  v += dpp_of<0x140>(v);  // row_mirror
  return v;
}
struct ScanStaging {
  __align__(16) float keys[2][GDN_SCAN_BLOCK][kDim], queries[2][GDN_SCAN_BLOCK][kDim];
  __align__(16) uint16_t values[2][GDN_SCAN_BLOCK][GDN_SCAN_STATE_ROWS], outputs[GDN_SCAN_BLOCK][GDN_SCAN_STATE_ROWS];
  float2 gates[2][GDN_SCAN_BLOCK];   // decay, beta
};
// One head's state rows rowBase .. + GDN_SCAN_STATE_ROWS - 1 through the run, by the first 256 threads of a workgroup.
// It passes scan_barriers(tokens) barriers.
__device__ __forceinline__ uint32_t scan_barriers(uint32_t tokens) { return 1u + 2u * ((tokens + GDN_SCAN_BLOCK - 1u) / GDN_SCAN_BLOCK); }
__device__ __forceinline__ void scan_state_rows(ScanStaging &staging, const uint16_t *__restrict__ queries, const uint16_t *__restrict__ keys,
                                                const uint16_t *__restrict__ values, const float *__restrict__ decay,
                                                const uint16_t *__restrict__ beta, uint8_t *__restrict__ states,
                                                uint16_t *__restrict__ recurrent_rows, const GdnPrefillParams &p, uint32_t head, uint32_t rowBase) {
  constexpr uint32_t B = GDN_SCAN_BLOCK, R = GDN_SCAN_STATE_ROWS, kPieces = R / 8;
  static_assert(B * kDim * 2 == 256 * 16, "a thread stages sixteen bytes of a block's keys and of its queries");
  static_assert(R == 16, "four waves of four rows hold a workgroup's state rows");
  auto &sk = staging.keys, &sq = staging.queries;
  auto &sv = staging.values;
  auto &so = staging.outputs;
  auto &gates = staging.gates;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const GdnShapeParams &s = p.shape;
  const uint32_t keyHead = head / (s.value_heads / s.key_heads), keyWidth = s.key_heads * kDim, valueWidth = s.value_heads * kDim;
  const uint32_t local = wave * 4u + (lane >> 4), column = 8u * (lane & 15u), tokens = p.tokens;
  const float *stateIn = reinterpret_cast<const float *>(states + p.current_cell + p.convolution_state_bytes + uint64_t(p.layer) * p.recurrent_layer_bytes);
  float *stateOut = reinterpret_cast<float *>(states + p.next_cell + p.convolution_state_bytes + uint64_t(p.layer) * p.recurrent_layer_bytes);
  const size_t stateAt = (size_t(head) * kDim + rowBase + local) * kDim + column;
  float state[2][4];
#pragma unroll
  for (uint32_t h = 0; h < 2; ++h) {
    const float4 loaded = *reinterpret_cast<const float4 *>(stateIn + stateAt + 4u * h);
    state[h][0] = loaded.x;
    state[h][1] = loaded.y;
    state[h][2] = loaded.z;
    state[h][3] = loaded.w;
  }
  // Rows at or past `tokens` keep what the registers held and are staged as they are: the loop below stops at the
  // run's last token, so those slots are never read.
  uint4 keyFetch = make_uint4(0, 0, 0, 0), queryFetch = keyFetch, valueFetch = keyFetch;
  float decayFetch = 0.f;
  uint16_t betaFetch = 0;
  auto fetch = [&](uint32_t start) __attribute__((always_inline)) {
    const uint32_t token = start + tid / 16u;
    if (token < tokens) {
      const size_t at = (size_t(p.first) + token) * keyWidth + keyHead * kDim + (tid % 16u) * 8u;
      keyFetch = *reinterpret_cast<const uint4 *>(keys + at);
      queryFetch = *reinterpret_cast<const uint4 *>(queries + at);
    }
    if (tid < kPieces * B && start + tid / kPieces < tokens)
      valueFetch = *reinterpret_cast<const uint4 *>(values + (size_t(p.first) + start + tid / kPieces) * valueWidth + head * kDim + rowBase + (tid % kPieces) * 8u);
    if (tid < B && start + tid < tokens) {
      decayFetch = decay[(size_t(p.first) + start + tid) * s.value_heads + head];
      betaFetch = beta[(size_t(p.first) + start + tid) * s.value_heads + head];
    }
  };
  auto widen = [&](float *to, const uint4 &v) __attribute__((always_inline)) {
    *reinterpret_cast<float4 *>(to) = make_float4(bf16_bits_to_float(v.x & 0xFFFFu), bf16_bits_to_float(v.x >> 16), bf16_bits_to_float(v.y & 0xFFFFu),
                                                  bf16_bits_to_float(v.y >> 16));
    *reinterpret_cast<float4 *>(to + 4) = make_float4(bf16_bits_to_float(v.z & 0xFFFFu), bf16_bits_to_float(v.z >> 16), bf16_bits_to_float(v.w & 0xFFFFu),
                                                      bf16_bits_to_float(v.w >> 16));
  };
  auto stage = [&](uint32_t buffer) __attribute__((always_inline)) {
    widen(&sk[buffer][tid / 16u][(tid % 16u) * 8u], keyFetch);
    widen(&sq[buffer][tid / 16u][(tid % 16u) * 8u], queryFetch);
    if (tid < kPieces * B) *reinterpret_cast<uint4 *>(&sv[buffer][tid / kPieces][(tid % kPieces) * 8u]) = valueFetch;
    if (tid < B) gates[buffer][tid] = make_float2(decayFetch, bf16_bits_to_float(betaFetch));
  };
  fetch(0);
  stage(0);
  __syncthreads();
  for (uint32_t start = 0, buffer = 0; start < tokens; start += B, buffer ^= 1u) {
    const bool more = start + B < tokens;
    if (more) fetch(start + B);
    const uint32_t count = min(B, tokens - start);
    // A token's operands leave LDS one token ahead of their use.
    struct Operands {
      float4 key[2], query[2];
      float2 gate;
      uint32_t value;
    };
    auto operands = [&](uint32_t t) __attribute__((always_inline)) {
      Operands o;
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) {
        o.key[h] = *reinterpret_cast<const float4 *>(&sk[buffer][t][column + 4u * h]);
        o.query[h] = *reinterpret_cast<const float4 *>(&sq[buffer][t][column + 4u * h]);
      }
      o.gate = gates[buffer][t];
      o.value = sv[buffer][t][local];
      return o;
    };
    static_assert(B == 16, "a row's sixteen lanes keep a block's outputs");
    float outputs = 0.f;
    Operands ahead = operands(0);
    auto step = [&](uint32_t t) __attribute__((always_inline)) {
      const Operands now = ahead;
      ahead = operands(min(t + 1u, B - 1u));  // past the block's last token: a staged slot nobody uses
      float memory[2], output[2];
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) {
        const float k[4] = {now.key[h].x, now.key[h].y, now.key[h].z, now.key[h].w};
        memory[h] = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          state[h][i] *= now.gate.x;
          memory[h] += state[h][i] * k[i];
        }
      }
      const float delta = (bf16_bits_to_float(now.value) - sixteen_sum(memory[0] + memory[1])) * now.gate.y;
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) {
        const float k[4] = {now.key[h].x, now.key[h].y, now.key[h].z, now.key[h].w};
        const float q[4] = {now.query[h].x, now.query[h].y, now.query[h].z, now.query[h].w};
        output[h] = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          state[h][i] += k[i] * delta;
          output[h] += state[h][i] * q[i];
        }
      }
      // lane t of a row's sixteen keeps token t's output
      const float sum = sixteen_sum(output[0] + output[1]);
      outputs = (lane & 15u) == t ? sum : outputs;
    };
    if (count == B) {
#pragma unroll
      for (uint32_t t = 0; t < B; ++t) step(t);
    } else {
      for (uint32_t t = 0; t < count; ++t) step(t);
    }
    so[lane & 15u][local] = uint16_t(float_to_bf16_bits(outputs));
    __syncthreads();  // the block's outputs are whole, and no wave reads its staged rows any more
    if (tid < kPieces * count)
      *reinterpret_cast<uint4 *>(recurrent_rows + (size_t(p.first) + start + tid / kPieces) * valueWidth + head * kDim + rowBase + (tid % kPieces) * 8u) =
          *reinterpret_cast<const uint4 *>(&so[tid / kPieces][(tid % kPieces) * 8u]);
    if (more) stage(buffer ^ 1u);
    __syncthreads();
  }
#pragma unroll
  for (uint32_t h = 0; h < 2; ++h)
    *reinterpret_cast<float4 *>(stateOut + stateAt + 4u * h) = make_float4(state[h][0], state[h][1], state[h][2], state[h][3]);
}
__global__ __launch_bounds__(256) void gdn_prefill_scan(const uint16_t *__restrict__ queries, const uint16_t *__restrict__ keys,
                                                        const uint16_t *__restrict__ values, const float *__restrict__ decay,
                                                        const uint16_t *__restrict__ beta, uint8_t *__restrict__ states,
                                                        uint16_t *__restrict__ recurrent_rows, GdnPrefillParams p) {
  constexpr uint32_t kGroups = kDim / GDN_SCAN_STATE_ROWS;
  __shared__ ScanStaging staging;
  scan_state_rows(staging, queries, keys, values, decay, beta, states, recurrent_rows, p, blockIdx.x / kGroups, (blockIdx.x % kGroups) * GDN_SCAN_STATE_ROWS);
}
SP_REGISTER_KERNEL("gdn_prefill_scan", &gdn_prefill_scan);

// ---- prefill in blocks of sixteen tokens, on the matrix cores ----
//
// Within a block that starts from the state S, with g_t the decay from its start to row t and D_tj that from row j to row t,
// the state after row t is g_t S + sum_{j <= t} D_tj u_j k_j', where the corrections u solve the triangular system
//   u_t + beta_t sum_{j < t} D_tj (k_t . k_j) u_j = beta_t (v_t - g_t S k_t).
// Its inverse (with the betas folded in, T) and the products A_tj = D_tj (q_t . k_j) of the outputs
//   o_t = g_t S q_t + sum_{j <= t} A_tj u_j
// depend on the block's rows alone: gdn_prefill_blocks works them out for every block at once, and what is left to do in
// order, gdn_prefill_block_scan, is per block two products with the state, one with T and the state's update, all MFMAs.
// (The chunkwise form of the gated delta rule: Yang, Kautz and Hatamizadeh, Gated Delta Networks, 2024, after Yang et al.,
// Parallelizing Linear Transformers with the Delta Rule over Sequence Length, 2024; here with the system solved per block.)
// A token is one dependent chain in gdn_prefill_scan (0.2 us each); here sixteen are: 2048 tokens of 16 / 32 heads 402 us
// there, 13 + 93 us here (0.72 us a block). The sums' order differs from the fold's, so a chunk through these kernels leaves
// the accepted blocks' cell to rounding, not bit for bit.
// Precision: keys and queries are bf16, as they are; the state and the corrections enter their products as three bf16 parts
// each, which hold all 24 bits, and every sum is fp32. Against 64-bit arithmetic the state of 32 heads is off by 5.0e-8 of
// its norm where the scan's is by 5.7e-8, and the rows by the same rounding to bf16 (tests/test_gdn_blocks_gpu.py).
// Values that are not finite: in these products a row of them would reach the rows of its block before it (the triangle's
// zeros multiply it) and an infinite state would be NaN (its parts are inf - inf). Either stays in the state's row to the
// run's end, where a workgroup that finds one in its rows takes the run again token by token, as the scan does and bit for
// bit. (A query that is not finite reaches its own output alone, here as there.)
__device__ __forceinline__ uint32_t upper_halves(float low, float high) {
  return __builtin_amdgcn_perm(__float_as_uint(high), __float_as_uint(low), 0x07060302u);
}
__device__ __forceinline__ float cut(float v) { return __uint_as_float(__float_as_uint(v) & 0xFFFF0000u); }
// Two values as three pairs of bf16 whose sums they are (each part the eight leading bits of what is left).
__device__ __forceinline__ void split3(float a, float b, uint32_t &high, uint32_t &middle, uint32_t &low) {
  high = upper_halves(a, b);
  const float a1 = a - cut(a), b1 = b - cut(b);
  middle = upper_halves(a1, b1);
  low = upper_halves(a1 - cut(a1), b1 - cut(b1));
}

// gdn_prefill_blocks: grid (value_heads, ceil(blocks / 4)), 256 threads, a wave per (block, value head). A run's last block
// may be short: rows past it repeat the last one with a decay of 1 and a beta of 0, which makes their corrections zero.
__global__ __launch_bounds__(256) void gdn_prefill_blocks(const uint16_t *__restrict__ queries, const uint16_t *__restrict__ keys,
                                                          const float *__restrict__ decay, const uint16_t *__restrict__ beta,
                                                          uint8_t *__restrict__ work, GdnPrefillParams p) {
  constexpr uint32_t B = GDN_SCAN_BLOCK;
  __shared__ __align__(16) uint16_t stagedKeys[4][B][kDim + 8];
  __shared__ __align__(16) float system[4][B][B];
  __shared__ __align__(16) float gates[4][2][B];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, row = lane & 15u, kq = lane >> 4;
  const GdnShapeParams s = p.shape;
  const uint32_t head = blockIdx.x, block = blockIdx.y * 4u + wave, start = block * B;
  const uint32_t perKey = s.value_heads / s.key_heads, keyHead = head / perKey, keyWidth = s.key_heads * kDim;
  if (start >= p.tokens) return;   // (no barrier below: a wave's LDS is its own)
  const uint32_t token = min(start + row, p.tokens - 1u);
  const size_t at = (size_t(p.first) + token) * keyWidth + keyHead * kDim + 8u * kq;
  uint4 key[4], query[4];
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w) {
    key[w] = *reinterpret_cast<const uint4 *>(keys + at + 32u * w);
    query[w] = *reinterpret_cast<const uint4 *>(queries + at + 32u * w);
  }
  if (kq == 0) {
    const size_t gate = (size_t(p.first) + token) * s.value_heads + head;
    const bool live = start + row < p.tokens;
    gates[wave][0][row] = live ? decay[gate] : 1.f;
    gates[wave][1][row] = live ? bf16_bits_to_float(beta[gate]) : 0.f;
  }
  // rows t = 4 kq + i, columns j = row
  f32x4 kk = {0.f, 0.f, 0.f, 0.f}, qk = kk;
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w) {
    kk = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(key[w]), as_bf16x8(key[w]), kk, 0, 0, 0);
    qk = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(query[w]), as_bf16x8(key[w]), qk, 0, 0, 0);
  }
  wave_lds_fence();
  float between[4], sinceStart[4], toEnd = 1.f, running = 1.f;
#pragma unroll
  for (uint32_t t = 0; t < B; ++t) {
    const float d = gates[wave][0][t];
    toEnd = t > row ? toEnd * d : 1.f;
    running *= d;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i)
      if (4u * kq + i == t) {
        between[i] = toEnd;
        sinceStart[i] = running;
      }
  }
  float *terms = reinterpret_cast<float *>(work) + (size_t(block) * s.value_heads + head) * GDN_BLOCK_TERMS;
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    const uint32_t t = 4u * kq + i;
    system[wave][t][row] = t > row ? gates[wave][1][t] * (between[i] * kk[i]) : 0.f;
    terms[B * B + t * B + row] = t >= row ? between[i] * qk[i] : 0.f;
    if (row == 0) {
      terms[2 * B * B + t] = sinceStart[i];
      terms[2 * B * B + 3 * B + t] = sinceStart[i] * gates[wave][1][t];
    }
  }
  if (kq == 0) {
    terms[2 * B * B + B + row] = toEnd;
    terms[2 * B * B + 2 * B + row] = gates[wave][1][row];
  }
  wave_lds_fence();
  // column j = row of the inverse, top down
  float x[B];
#pragma unroll
  for (uint32_t t = 0; t < B; ++t) {
    float sum = t == row ? 1.f : 0.f;
#pragma unroll
    for (uint32_t j = 0; j < t; ++j) sum = __fmaf_rn(-system[wave][t][j], x[j], sum);
    x[t] = sum;
    if (kq == t / 4u) terms[t * B + row] = t == row ? 0.f : sum;
  }
  if (head % perKey) return;
  // The keys as the update's operands: lane (r, kq) of wave w's tile m holds tokens 4 kq .. + 3 of dimension
  // 32 w + 8 (r / 4) + 4 m + r % 4, the dimension that row r of the tile's part of the state holds, twice over: the update
  // multiplies them by the corrections' leading parts and by what is left of those.
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w) *reinterpret_cast<uint4 *>(&stagedKeys[wave][row][32u * w + 8u * kq]) = key[w];
  wave_lds_fence();
  uint4 *out = reinterpret_cast<uint4 *>(work + gdn_prefill_block_keys_offset(p.tokens, s.value_heads) +
                                         (size_t(block) * s.key_heads + keyHead) * GDN_BLOCK_KEYS_BYTES);
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w) {
#pragma unroll
    for (uint32_t m = 0; m < 2; ++m) {
      const uint32_t dimension = 32u * w + 8u * (row >> 2) + 4u * m + (row & 3u);
      uint32_t words[2];
#pragma unroll
      for (uint32_t e = 0; e < 2; ++e)
        words[e] = uint32_t(stagedKeys[wave][4u * kq + 2u * e][dimension]) | (uint32_t(stagedKeys[wave][4u * kq + 2u * e + 1u][dimension]) << 16);
      out[w * 128u + m * 64u + lane] = make_uint4(words[0], words[1], words[0], words[1]);
    }
  }
}
SP_REGISTER_KERNEL("gdn_prefill_blocks", &gdn_prefill_blocks);

// gdn_prefill_block_scan: grid (value_heads * 8), 320 threads. A workgroup carries sixteen rows (value dimensions) of a head's
// state through the run's blocks. Four waves hold it, wave w the key dimensions 32 w .. + 31: lane (r, kq) row r's dimensions
// 32 w + 8 kq .. + 7, which are both the result of the update and, cut in three, the operand of the next block's products, so
// the state never moves between lanes. Their shares of S k and S q meet in LDS, one barrier a block; every wave then solves
// for all sixteen rows' corrections (four fp32 MFMAs), the four update their columns and the fifth writes the outputs. What a
// block needs from memory is in flight three blocks ahead (all of it issued at a block's end: 113 us, the compiler's own order:
// 124; the outputs by the four waves in turn: 118). One workgroup a compute unit: the pass is the latency of a block's
// chain. The workgroups of a head read the same keys and terms: head h's run on die h % 8 (workgroup b runs on die b % 8)
// wherever the heads fill the dies.
struct BlockTerms {
  uint4 solve, started, weight;   // of rows `row` (solve), 4 kq .. + 3
  uint32_t value[4];              // of token 4 kq + i, value dimensions rowBase + (row & ~1) and the next
};
__global__ __launch_bounds__(320, 1) void gdn_prefill_block_scan(const uint16_t *__restrict__ queries, const uint16_t *__restrict__ keys,
                                                                 const uint16_t *__restrict__ values, const float *__restrict__ decay,
                                                                 const uint16_t *__restrict__ beta, const uint8_t *__restrict__ work,
                                                                 uint8_t *__restrict__ states, uint16_t *__restrict__ recurrent_rows,
                                                                 GdnPrefillParams p) {
  constexpr uint32_t B = GDN_SCAN_BLOCK, kAhead = 4;
  __shared__ __align__(16) float4 shares[2][2][4][64];   // [block parity][S k, S q][wave][lane]
  __shared__ ScanStaging staging;                        // of the run again
  __shared__ uint32_t unbounded;                         // the state after the run is not finite
  const uint32_t tid = threadIdx.x, lane = tid & 63u, row = lane & 15u, kq = lane >> 4;
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
  const GdnShapeParams s = p.shape;
  if (tid == 0) unbounded = 0;   // (set behind the blocks' barriers)
  const uint32_t head = blockIdx.x % s.value_heads, rowBase = blockIdx.x / s.value_heads * 16u;
  const uint32_t keyHead = head / (s.value_heads / s.key_heads), keyWidth = s.key_heads * kDim, valueWidth = s.value_heads * kDim;
  const uint32_t blocks = (p.tokens + B - 1u) / B, rounds = (blocks + kAhead - 1u) / kAhead;
  // Every stream through a buffer resource of the run's rows: rows past them, and blocks past the last, read as zeros (which
  // correct nothing), and writes there go nowhere.
  const uint32_t keyRow = keyWidth * 2u, valueRow = valueWidth * 2u, keysAt = uint32_t(gdn_prefill_block_keys_offset(p.tokens, s.value_heads));
  const uint32_t termsBlock = s.value_heads * (GDN_BLOCK_TERMS * 4u), keysBlock = s.key_heads * GDN_BLOCK_KEYS_BYTES;
  const Resource valueRows = make_resource(values + size_t(p.first) * valueWidth, p.tokens * valueRow);
  const Resource terms = make_resource(work, blocks * termsBlock);
  uint32_t valueAt[4];
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) valueAt[i] = (4u * kq + i) * valueRow + (head * kDim + rowBase + (row & ~1u)) * 2u;
  uint32_t termAt = head * (GDN_BLOCK_TERMS * 4u) + (row * B + 4u * kq) * 4u, rowsAt = head * (GDN_BLOCK_TERMS * 4u) + 2u * B * B * 4u + 16u * kq;
  auto fetchValues = [&](BlockTerms &f) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) f.value[i] = __builtin_amdgcn_raw_buffer_load_b32(valueRows, int(valueAt[i]), 0, 0);
  };
  auto fetchSolve = [&](BlockTerms &f) __attribute__((always_inline)) { f.solve = load128<0>(terms, termAt); };
  auto fetchWeights = [&](BlockTerms &f) __attribute__((always_inline)) {
    f.weight = load128<0>(terms, rowsAt + 2u * B * 4u);
    f.started = load128<0>(terms, rowsAt + 3u * B * 4u);
  };
  auto advanceTerms = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) valueAt[i] += B * valueRow;
    termAt += termsBlock;
    rowsAt += termsBlock;
  };
  // A fetched word where it is used: what is computed from it, and with that the wait for it, stays there.
  auto used = [](uint32_t v) __attribute__((always_inline)) {
    asm volatile("" : "+v"(v));
    return v;
  };
  auto floats = [](const uint4 &v) __attribute__((always_inline)) { return __builtin_bit_cast(f32x4, v); };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  auto whole = [&](uint32_t parity, uint32_t which) __attribute__((always_inline)) {   // the waves' shares added
    f32x4 part[4], sum;
#pragma unroll
    for (uint32_t w = 0; w < 4; ++w) part[w] = __builtin_bit_cast(f32x4, shares[parity][which][w][lane]);
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) sum[i] = (part[0][i] + part[1][i]) + (part[2][i] + part[3][i]);
    return sum;
  };
  const uint32_t valueShift = row & 1u ? 0u : 16u;
  // `between(i)` is issued behind the i-th product, each of which waits for the one before.
  auto correctionsOf = [&](const BlockTerms &f, const f32x4 &memory, auto &&between) __attribute__((always_inline)) {
    const f32x4 solve = floats(f.solve), started = floats(f.started), weight = floats(f.weight);
    f32x4 own, sum = zero;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i)
      // (the last product is exact)
      own[i] = __fmaf_rn(-started[i], memory[i], weight[i] * __uint_as_float((used(f.value[i]) << valueShift) & 0xFFFF0000u));
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {   // token 4 kq + i in place kq
      sum = __builtin_amdgcn_mfma_f32_16x16x4f32(solve[i], own[i], sum, 0, 0, 0);
      between(i);
    }
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) sum[i] += own[i];
    return sum;
  };
  // (A block's shares are written over those of two blocks before, which every wave has read once it is past the barrier of
  // the block between. Both kinds of wave below pass rounds * kAhead barriers, one that ends the run, and those of the run
  // again where there is one.)
  if (wave == 4u) {
    const Resource outputRows = make_resource(recurrent_rows + size_t(p.first) * valueWidth, p.tokens * valueRow);
    struct Fetched {
      BlockTerms terms;
      uint4 outputs, sinceStart;
    };
    uint32_t outputAt[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) outputAt[i] = valueAt[i] + (row & 1u) * 2u;
    auto fetch = [&](Fetched &f) __attribute__((always_inline)) {
      fetchValues(f.terms);
      fetchSolve(f.terms);
      fetchWeights(f.terms);
      f.sinceStart = load128<0>(terms, rowsAt);
      f.outputs = load128<0>(terms, termAt + B * B * 4u);
      advanceTerms();
    };
    auto run = [&](uint32_t parity, const Fetched &f) __attribute__((always_inline)) {
      __syncthreads();
      const f32x4 memory = whole(parity, 0);
      f32x4 out = whole(parity, 1);
      const f32x4 corrections = correctionsOf(f.terms, memory, [](uint32_t) {}), sinceStart = floats(f.sinceStart), outputs = floats(f.outputs);
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) out[i] *= sinceStart[i];
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) out = __builtin_amdgcn_mfma_f32_16x16x4f32(outputs[i], corrections[i], out, 0, 0, 0);
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, static_cast<__bf16>(out[i])), outputRows, int(outputAt[i]), 0, 0);
        outputAt[i] += B * valueRow;
      }
    };
    Fetched ahead[kAhead];
#pragma unroll
    for (uint32_t a = 0; a < kAhead; ++a) {
      fetch(ahead[a]);
      __builtin_amdgcn_sched_barrier(0);   // (in the order the loop waits for them)
    }
    for (uint32_t round = 0, parity = 0; round < rounds; ++round) {
#pragma unroll
      for (uint32_t a = 0; a < kAhead; ++a, parity ^= 1u) {
        run(parity, ahead[a]);
        __builtin_amdgcn_sched_barrier(0);
        fetch(ahead[a]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
    if (unbounded) {
      __threadfence();   // (this run's outputs are out before the run again stores its first, behind two more barriers)
      for (uint32_t n = scan_barriers(p.tokens); n; --n) __syncthreads();
    }
    return;
  }
  const float *stateIn = reinterpret_cast<const float *>(states + p.current_cell + p.convolution_state_bytes + uint64_t(p.layer) * p.recurrent_layer_bytes);
  float *stateOut = reinterpret_cast<float *>(states + p.next_cell + p.convolution_state_bytes + uint64_t(p.layer) * p.recurrent_layer_bytes);
  const size_t stateAt = (size_t(head) * kDim + rowBase + row) * kDim + 32u * wave + 8u * kq;
  f32x4 state[2];
#pragma unroll
  for (uint32_t m = 0; m < 2; ++m) state[m] = *reinterpret_cast<const f32x4 *>(stateIn + stateAt + 4u * m);
  const Resource keyRows = make_resource(keys + size_t(p.first) * keyWidth, p.tokens * keyRow);
  const Resource queryRows = make_resource(queries + size_t(p.first) * keyWidth, p.tokens * keyRow);
  const Resource operands = make_resource(work + keysAt, blocks * keysBlock);
  uint32_t keyAt = row * keyRow + (keyHead * kDim + 32u * wave + 8u * kq) * 2u, operandAt = keyHead * GDN_BLOCK_KEYS_BYTES + wave * 2048u + lane * 16u;
  uint32_t decayAt = head * (GDN_BLOCK_TERMS * 4u) + (2u * B * B + B - 1u) * 4u;
  struct Fetched {
    BlockTerms terms;
    uint4 key, query;             // this wave's 32 dimensions of token `row`
    uint4 update[2];              // and of tokens 4 kq .. + 3, twice over
    uint4 toEnd;
    uint32_t decay;               // the whole block's
  };
  // The next block's loads in six pieces, which leave between the products of a block: all at once they fill the address
  // unit that the four waves share, and a wave that waits there runs nothing else.
  auto fetch = [&](Fetched &f, uint32_t piece) __attribute__((always_inline)) {
    if (piece == 0) {
      f.key = load128<0>(keyRows, keyAt);
      f.query = load128<0>(queryRows, keyAt);
      keyAt += B * keyRow;
    } else if (piece == 1) {
      fetchSolve(f.terms);
    } else if (piece == 2) {
      fetchWeights(f.terms);
    } else if (piece == 3) {
      fetchValues(f.terms);
    } else if (piece == 4) {
      f.toEnd = load128<0>(terms, rowsAt + B * 4u);
      f.decay = __builtin_amdgcn_raw_buffer_load_b32(terms, int(decayAt), 0, 0);
      advanceTerms();
      decayAt += termsBlock;
    } else {
#pragma unroll
      for (uint32_t m = 0; m < 2; ++m) f.update[m] = load128<0>(operands, operandAt + 1024u * m);
      operandAt += keysBlock;
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto run = [&](uint32_t block, uint32_t parity, const Fetched &f, Fetched &next) __attribute__((always_inline)) {
    uint32_t high[4], middle[4], low[4];
#pragma unroll
    for (uint32_t e = 0; e < 4; ++e) split3(state[e >> 1][2u * (e & 1u)], state[e >> 1][2u * (e & 1u) + 1u], high[e], middle[e], low[e]);
    const bf16x8 parts[3] = {as_bf16x8(make_uint4(low[0], low[1], low[2], low[3])), as_bf16x8(make_uint4(middle[0], middle[1], middle[2], middle[3])),
                             as_bf16x8(make_uint4(high[0], high[1], high[2], high[3]))};
    f32x4 sk = zero, sq = zero;   // rows are tokens 4 kq + i, column `row` a value dimension
#pragma unroll
    for (uint32_t e = 0; e < 3; ++e) {
      sk = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(f.key), parts[e], sk, 0, 0, 0);
      sq = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(f.query), parts[e], sq, 0, 0, 0);
    }
    shares[parity][0][wave][lane] = __builtin_bit_cast(float4, sk);
    shares[parity][1][wave][lane] = __builtin_bit_cast(float4, sq);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    fetch(next, 0);
    const f32x4 corrections = correctionsOf(f.terms, whole(parity, 0), [&](uint32_t i) __attribute__((always_inline)) { fetch(next, 1u + i); });
    const f32x4 toEnd = floats(f.toEnd);
    // the update: places 0..3 of an operand's eight the corrections' leading parts, and apart from them the two parts left
    uint32_t uh[2], um[2], ul[2];
#pragma unroll
    for (uint32_t e = 0; e < 2; ++e)
      split3(corrections[2u * e] * toEnd[2u * e], corrections[2u * e + 1u] * toEnd[2u * e + 1u], uh[e], um[e], ul[e]);
    const bf16x8 leading = as_bf16x8(make_uint4(uh[0], uh[1], 0u, 0u)), last = as_bf16x8(make_uint4(um[0], um[1], ul[0], ul[1]));
    const float kept = block < blocks ? __uint_as_float(f.decay) : 1.f;
#pragma unroll
    for (uint32_t m = 0; m < 2; ++m) {
      const bf16x8 key = as_bf16x8(f.update[m]);
      const f32x4 most = __builtin_amdgcn_mfma_f32_16x16x32_bf16(key, leading, zero, 0, 0, 0);
      const f32x4 rest = __builtin_amdgcn_mfma_f32_16x16x32_bf16(key, last, zero, 0, 0, 0);
      if (m == 0) fetch(next, 5);
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) state[m][i] = __fmaf_rn(state[m][i], kept, rest[i]) + most[i];
    }
  };
  Fetched ahead[kAhead];
#pragma unroll
  for (uint32_t a = 0; a + 1 < kAhead; ++a)
#pragma unroll
    for (uint32_t piece = 0; piece < 6; ++piece) fetch(ahead[a], piece);   // (in the order the loop waits for them)
  for (uint32_t round = 0, parity = 0; round < rounds; ++round) {
#pragma unroll
    for (uint32_t a = 0; a < kAhead; ++a, parity ^= 1u) {
      run(round * kAhead + a, parity, ahead[a], ahead[(a + kAhead - 1u) % kAhead]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  uint32_t most = 0;   // the magnitudes' bits order as the magnitudes do, those past the infinity's are NaNs
#pragma unroll
  for (uint32_t m = 0; m < 2; ++m)
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) most = max(most, __float_as_uint(state[m][i]) & 0x7FFFFFFFu);
  if (most >= 0x7F800000u) unbounded = 1;
  __syncthreads();
  if (unbounded) {
    scan_state_rows(staging, queries, keys, values, decay, beta, states, recurrent_rows, p, head, rowBase);
    return;
  }
#pragma unroll
  for (uint32_t m = 0; m < 2; ++m) *reinterpret_cast<f32x4 *>(stateOut + stateAt + 4u * m) = state[m];
}
SP_REGISTER_KERNEL("gdn_prefill_block_scan", &gdn_prefill_block_scan);

// gdn_prefill_gate: grid (value_heads, ceil(tokens / (4 GDN_GATE_ROWS))), 256 threads, a wave per GDN_GATE_ROWS rows of a
// value head: the gated output norm of the scan's rows (prefill/gdn.metal:312-341, gdn.metal:489-526). A wave of one row
// only waited for its four loads: 2048 rows of 32 heads 28 us so, 17.6 with the rows' loads out together.
__global__ __launch_bounds__(256) void gdn_prefill_gate(const uint16_t *__restrict__ recurrent_rows, const uint16_t *__restrict__ packed,
                                                        const void *__restrict__ norm_weight, uint16_t *__restrict__ hidden,
                                                        GdnPrefillParams p) {
  constexpr uint32_t R = GDN_GATE_ROWS;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, head = blockIdx.x, firstRow = (blockIdx.y * 4u + wave) * R;
  if (firstRow >= p.tokens) return;
  const uint32_t rows = min(R, p.tokens - firstRow);
  const size_t first = size_t(p.first) + firstRow;
  const GdnShapeParams s = p.shape;
  const uint32_t perKey = s.value_heads / s.key_heads, valueWidth = s.value_heads * kDim;
  const uint32_t outHead = (p.flags & GDN_TILED_HEADS) ? (head % perKey) * s.key_heads + head / perKey : head;
  float value[R][2], z[R][2], weight[2];
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    const size_t token = first + min(r, rows - 1u);   // the last row again past the run's end
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part) {
      value[r][part] = bf16_bits_to_float(recurrent_rows[token * valueWidth + head * kDim + lane + 64u * part]);
      z[r][part] = bf16_bits_to_float(packed[token * s.packed_width + s.conv_dim + head * kDim + lane + 64u * part]);
    }
  }
#pragma unroll
  for (uint32_t part = 0; part < 2; ++part) weight[part] = norm_weight_of(norm_weight, p.flags, lane + 64u * part);
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    if (r >= rows) break;
    uint32_t gated[2];
    gated_values(value[r], weight, z[r], p.flags, gated);
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part)
      hidden[((first + r) * s.value_heads + outHead) * kDim + lane + 64u * part] = uint16_t(gated[part]);
  }
}
SP_REGISTER_KERNEL("gdn_prefill_gate", &gdn_prefill_gate);

// gdn_prefill_gate_table: grid (64 * ceil(16 tiles / 64)), 256 threads, a workgroup a row of the chunk's wide table: the row's
// gated heads, a wave every fourth one, eight heads' loads out together, meet in LDS and leave as the table the output
// projection reads. The values and the table are the bits of gdn_prefill_gate and gguf_wide_table, whose rows between them
// went to memory and back: 2048 rows of 32 heads 18.0 + 11.4 us in the two, 21.4 here (21.9 with four heads' loads out). Bound
// by memory and what follows it in a row's workgroup, the sums and the scale. Up to GDN_GATE_TABLE_WIDTH values a row, 16 KB
// of LDS: what the norms' tables hold; wider rows and an odd number of heads (half a super-block) take the two.
__global__ __launch_bounds__(256) void gdn_prefill_gate_table(const uint16_t *__restrict__ recurrent_rows, const uint16_t *__restrict__ packed,
                                                              const void *__restrict__ norm_weight, uint8_t *__restrict__ table,
                                                              GdnPrefillParams p) {
  constexpr uint32_t R = 8;
  __shared__ __align__(16) uint16_t gatedRow[GDN_GATE_TABLE_WIDTH];
  const GdnShapeParams s = p.shape;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, row = wide_table_row_of(blockIdx.x);
  const uint32_t tiles = gguf_wide_tiles(p.tokens), perKey = s.value_heads / s.key_heads, valueWidth = s.value_heads * kDim;
  if (row >= 16u * tiles || valueWidth > GDN_GATE_TABLE_WIDTH) return;
  const bool live = row < p.tokens;
  if (live) {
    const uint16_t *values = recurrent_rows + size_t(row) * valueWidth, *gates = packed + size_t(row) * s.packed_width + s.conv_dim;
    float weight[2];
#pragma unroll
    for (uint32_t part = 0; part < 2; ++part) weight[part] = norm_weight_of(norm_weight, p.flags, lane + 64u * part);
    for (uint32_t first = wave; first < s.value_heads; first += 4u * R) {
      float value[R][2], z[R][2];
#pragma unroll
      for (uint32_t r = 0; r < R; ++r) {
        const uint32_t head = min(first + 4u * r, s.value_heads - 1u);
#pragma unroll
        for (uint32_t part = 0; part < 2; ++part) {
          value[r][part] = bf16_bits_to_float(values[head * kDim + lane + 64u * part]);
          z[r][part] = bf16_bits_to_float(gates[head * kDim + lane + 64u * part]);
        }
      }
#pragma unroll
      for (uint32_t r = 0; r < R; ++r) {
        const uint32_t head = first + 4u * r;
        if (head >= s.value_heads) break;
        const uint32_t outHead = (p.flags & GDN_TILED_HEADS) ? (head % perKey) * s.key_heads + head / perKey : head;
        uint32_t gated[2];
        gated_values(value[r], weight, z[r], p.flags, gated);
#pragma unroll
        for (uint32_t part = 0; part < 2; ++part) gatedRow[outHead * kDim + lane + 64u * part] = uint16_t(gated[part]);
      }
    }
  }
  __syncthreads();
  const GgufWideTableParams t{valueWidth, 1u, tiles, 0u};
  uint4 *entries = reinterpret_cast<uint4 *>(table + row / 16u * gguf_wide_tile_bytes(valueWidth)) + row % 16u;
  const float scale = wide_table_row<false, 4, 4>(gatedRow, nullptr, t, live ? 0u : 1u, [&](uint32_t line, uint32_t, uint32_t, uint4 entry)
                                                  __attribute__((always_inline)) { entries[size_t(line) * 16u] = entry; });
  if (threadIdx.x == 0) wide_scales_of(table, t)[row] = scale;
}
SP_REGISTER_KERNEL("gdn_prefill_gate_table", &gdn_prefill_gate_table);

} // namespace splash::kernels
