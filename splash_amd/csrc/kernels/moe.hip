// Mixture-of-experts routing around the grouped expert projections (kernels/gguf_linear.hip):
// top-k selection, grouping of routes by expert, the tiles' activation tables, the weighted sum
// (the reference's kernels/shared/moe.metal).
#include "abi/Moe.h"
#include "backend/KernelRegistry.hpp"
#include "kernels/device_common.hpp"

namespace splash::kernels {

// moe_route_select (moe.metal:23-113): one wave per row; lane l holds experts l, l + 64, ... Each
// rank takes the highest remaining score and, among equals, the lowest expert id.
// A gated shared expert's weight is the sigmoid of the row's product with the scalar gate: lane l sums dimensions l,
// l + 64, ... in order, the lanes' sums add by the wave's exchanges at distances 32, 16, ... 1.
__global__ __launch_bounds__(64) void moe_route_select(const float *__restrict__ scores, const uint16_t *__restrict__ input,
                                                       const float *__restrict__ shared_gate, uint32_t *__restrict__ selected,
                                                       float *__restrict__ weights, MoeRouteParams p) {
  constexpr uint32_t kPerLane = MOE_MAXIMUM_EXPERTS / 64u;
  __shared__ float ordered[MOE_MAXIMUM_TOP];
  const uint32_t row = blockIdx.x, lane = threadIdx.x, perRow = p.top_k + p.shared;
  if (p.shared) {
    float weight = 1.0f;
    if (p.shared_gated) {
      const uint16_t *x = input + size_t(row) * p.input_size;
      float scalar = 0.f;
      for (uint32_t d = lane; d < p.input_size; d += 64u) scalar += bf16_bits_to_float(x[d]) * shared_gate[d];
      scalar = wave_sum(scalar);
      weight = 1.0f / (1.0f + __builtin_amdgcn_exp2f(-1.44269504089f * scalar));
    }
    if (lane < p.shared) {
      selected[size_t(row) * perRow + p.top_k + lane] = p.experts + lane;
      weights[size_t(row) * perRow + p.top_k + lane] = weight;
    }
  }
  float mine[kPerLane];
#pragma unroll
  for (uint32_t slot = 0; slot < kPerLane; ++slot) {
    const uint32_t expert = lane + 64u * slot;
    mine[slot] = expert < p.experts ? scores[size_t(row) * p.score_stride + expert] : -INFINITY;
  }
  for (uint32_t rank = 0; rank < p.top_k; ++rank) {
    float best = -INFINITY;
    uint32_t bestSlot = 0;
#pragma unroll
    for (uint32_t slot = 0; slot < kPerLane; ++slot)
      if (mine[slot] > best) {
        best = mine[slot];
        bestSlot = slot;
      }
    const float rowBest = wave_max(best);
    uint32_t candidate = best == rowBest ? lane + 64u * bestSlot : 0xFFFFFFFFu;
    uint32_t winner = candidate;
    winner = min(winner, lane_xor<32>(winner));
    winner = min(winner, lane_xor<16>(winner));
    winner = min(winner, lane_xor<8>(winner));
    winner = min(winner, lane_xor<4>(winner));
    winner = min(winner, lane_xor<2>(winner));
    winner = min(winner, lane_xor<1>(winner));
    if (candidate == winner) {
#pragma unroll
      for (uint32_t slot = 0; slot < kPerLane; ++slot)
        if (slot == bestSlot) mine[slot] = -INFINITY;
    }
    if (lane == 0) {
      ordered[rank] = rowBest;
      selected[size_t(row) * perRow + rank] = winner;
    }
  }
  __syncthreads();
  if (lane < p.top_k) {
    float denominator = 0.f;
    if (p.sigmoid_router) {
      const auto sigmoid = [](float x) { return 1.0f / (1.0f + __builtin_amdgcn_exp2f(-1.44269504089f * x)); };
      for (uint32_t other = 0; other < p.top_k; ++other) denominator += sigmoid(ordered[other]);
      weights[size_t(row) * perRow + lane] = sigmoid(ordered[lane]) / (denominator + 1e-20f);
    } else {
      for (uint32_t other = 0; other < p.top_k; ++other) denominator += __builtin_amdgcn_exp2f((ordered[other] - ordered[0]) * 1.44269504089f);
      weights[size_t(row) * perRow + lane] = __builtin_amdgcn_exp2f((ordered[lane] - ordered[0]) * 1.44269504089f) / denominator;
    }
  }
}
SP_REGISTER_KERNEL("moe_route_select", &moe_route_select);

// moe_group_routes: one workgroup of 1024 threads, work in proportion to the routes. Every route sets its bit
// in its expert's row of a bit matrix (an OR: whatever order the threads run in, the matrix is the same);
// a thread per expert counts its row word by word, which gives the expert's routes before each word and its
// tiles; a route's place among its expert's is then those before its word plus the set bits below its own, so
// an expert's routes keep their route order and the grouping never depends on timing.
__global__ __launch_bounds__(1024) void moe_group_routes(const uint32_t *__restrict__ selected, uint32_t *__restrict__ route_slot,
                                                         uint32_t *__restrict__ slot_row, uint32_t *__restrict__ tile_expert,
                                                         uint32_t *__restrict__ tile_rows, uint32_t *__restrict__ tile_total,
                                                         MoeGroupParams p) {
  __shared__ uint32_t masks[MOE_GROUP_WORDS];   // [expert][word]: bit b of word w: route 32 w + b is the expert's
  __shared__ uint16_t before[MOE_GROUP_WORDS];  // [expert][word]: the expert's routes before word w
  __shared__ uint32_t firstTile[MOE_MAXIMUM_EXPERTS], waveTiles[MOE_MAXIMUM_EXPERTS / 64u];
  constexpr uint32_t kMine = 256u * MOE_MAXIMUM_TOP / 1024u;  // routes a thread may own
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t words = (p.routes + 31u) / 32u;
  for (uint32_t i = tid; i < p.experts * words; i += 1024u) masks[i] = 0u;
  for (uint32_t slot = tid; slot < p.maximum_tiles * MOE_TILE_ROWS; slot += 1024u) slot_row[slot] = MOE_NO_ROW;
  uint32_t mine[kMine];
#pragma unroll
  for (uint32_t i = 0; i < kMine; ++i) {
    const uint32_t route = tid + 1024u * i;
    mine[i] = route < p.routes ? selected[route] : 0u;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t i = 0; i < kMine; ++i) {
    const uint32_t route = tid + 1024u * i;
    if (route < p.routes) atomicOr(&masks[mine[i] * words + route / 32u], 1u << (route % 32u));
  }
  __syncthreads();
  // The expert's routes in all, and before each word of its row.
  uint32_t total = 0;
  if (tid < p.experts)
    for (uint32_t w = 0; w < words; ++w) {
      before[tid * words + w] = uint16_t(total);
      total += uint32_t(__builtin_popcount(masks[tid * words + w]));
    }
  // First tiles: an exclusive sum of the experts' tile counts, by waves and then over the waves' sums.
  const uint32_t tiles = (total + MOE_TILE_ROWS - 1u) / MOE_TILE_ROWS;
  uint32_t running = tiles;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t up = uint32_t(__shfl_up(int(running), o, 64));
    if (lane >= uint32_t(o)) running += up;
  }
  if (lane == 63u && tid < MOE_MAXIMUM_EXPERTS) waveTiles[wave] = running;
  __syncthreads();
  if (tid < MOE_MAXIMUM_EXPERTS) {
    uint32_t start = 0;
    for (uint32_t w = 0; w < wave; ++w) start += waveTiles[w];
    firstTile[tid] = start + running - tiles;
    if (tid == MOE_MAXIMUM_EXPERTS - 1u) tile_total[0] = start + running;
    for (uint32_t t = 0; t < tiles; ++t) {
      tile_expert[firstTile[tid] + t] = tid;
      tile_rows[firstTile[tid] + t] = min(MOE_TILE_ROWS, total - t * MOE_TILE_ROWS);
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t i = 0; i < kMine; ++i) {
    const uint32_t route = tid + 1024u * i;
    if (route >= p.routes) continue;
    const uint32_t at = mine[i] * words + route / 32u;
    const uint32_t placed = before[at] + uint32_t(__builtin_popcount(masks[at] & ((1u << (route % 32u)) - 1u)));
    const uint32_t slot = (firstTile[mine[i]] + placed / MOE_TILE_ROWS) * MOE_TILE_ROWS + placed % MOE_TILE_ROWS;
    route_slot[route] = slot;
    slot_row[slot] = route / p.top_k;
  }
}
SP_REGISTER_KERNEL("moe_group_routes", &moe_group_routes);

// The chunk's grouping (abi/Moe.h). Counting is an LDS histogram; placing repeats moe_group_routes' bit matrix for a
// window's routes, offset by the expert's first slot and the windows before: both follow from the counts of every window,
// which each workgroup sums for itself.
__global__ __launch_bounds__(1024) void moe_chunk_count(const uint32_t *__restrict__ selected, uint32_t *__restrict__ counts, MoeChunkParams p) {
  __shared__ uint32_t bins[MOE_MAXIMUM_EXPERTS];
  const uint32_t tid = threadIdx.x, first = blockIdx.x * MOE_CHUNK_ROUTES, last = min(p.routes, first + MOE_CHUNK_ROUTES);
  if (tid < MOE_MAXIMUM_EXPERTS) bins[tid] = 0u;
  __syncthreads();
  for (uint32_t route = first + tid; route < last; route += 1024u) atomicAdd(&bins[selected[route]], 1u);
  __syncthreads();
  if (tid < p.experts) counts[blockIdx.x * p.experts + tid] = bins[tid];
}
SP_REGISTER_KERNEL("moe_chunk_count", &moe_chunk_count);

__global__ __launch_bounds__(1024) void moe_chunk_place(const uint32_t *__restrict__ selected, const uint32_t *__restrict__ counts,
                                                        uint32_t *__restrict__ route_slot, uint32_t *__restrict__ slot_row,
                                                        MoeChunkTask *__restrict__ tasks, uint32_t *__restrict__ totals, MoeChunkParams p) {
  constexpr uint32_t kWords = MOE_CHUNK_ROUTES / 32u, kMine = MOE_CHUNK_ROUTES / 1024u;
  __shared__ uint32_t masks[MOE_MAXIMUM_EXPERTS * kWords];
  __shared__ uint16_t before[MOE_MAXIMUM_EXPERTS * kWords];
  __shared__ uint32_t firstSlot[MOE_MAXIMUM_EXPERTS], waveTiles[MOE_MAXIMUM_EXPERTS / 64u], waveTasks[MOE_MAXIMUM_EXPERTS / 64u];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, window = blockIdx.x, windows = gridDim.x;
  const uint32_t firstRoute = window * MOE_CHUNK_ROUTES, mineCount = min(p.routes - firstRoute, MOE_CHUNK_ROUTES);
  for (uint32_t i = tid; i < p.experts * kWords; i += 1024u) masks[i] = 0u;
  uint32_t mine[kMine];
#pragma unroll
  for (uint32_t i = 0; i < kMine; ++i) mine[i] = tid + 1024u * i < mineCount ? selected[firstRoute + tid + 1024u * i] : 0u;
  // thread e: expert e's routes in all and in the windows before
  uint32_t total = 0, earlier = 0;
  if (tid < p.experts)
    for (uint32_t w = 0; w < windows; ++w) {
      const uint32_t c = counts[w * p.experts + tid];
      total += c;
      if (w < window) earlier += c;
    }
  const uint32_t tiles = (total + MOE_TILE_ROWS - 1u) / MOE_TILE_ROWS, parts = (tiles + p.task_tiles - 1u) / p.task_tiles;
  uint32_t runningTiles = tiles, runningTasks = parts;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t a = uint32_t(__shfl_up(int(runningTiles), o, 64)), b = uint32_t(__shfl_up(int(runningTasks), o, 64));
    if (lane >= uint32_t(o)) {
      runningTiles += a;
      runningTasks += b;
    }
  }
  if (lane == 63u && tid < MOE_MAXIMUM_EXPERTS) {
    waveTiles[wave] = runningTiles;
    waveTasks[wave] = runningTasks;
  }
  __syncthreads();
  if (tid < MOE_MAXIMUM_EXPERTS) {
    uint32_t tile = runningTiles - tiles, task = runningTasks - parts;
    for (uint32_t w = 0; w < wave; ++w) {
      tile += waveTiles[w];
      task += waveTasks[w];
    }
    firstSlot[tid] = tile * MOE_TILE_ROWS + earlier;
    if (window == 0) {
      for (uint32_t i = 0; i < parts; ++i) {
        const uint32_t from = tiles * i / parts, to = tiles * (i + 1u) / parts;
        tasks[task + i] = MoeChunkTask{tid, tile + from, to - from, 0u};
      }
      for (uint32_t slot = total; slot < tiles * MOE_TILE_ROWS; ++slot) slot_row[tile * MOE_TILE_ROWS + slot] = MOE_NO_ROW;
      if (tid == MOE_MAXIMUM_EXPERTS - 1u) {
        totals[0] = tile + tiles;
        totals[1] = task + parts;
      }
    }
  }
#pragma unroll
  for (uint32_t i = 0; i < kMine; ++i) {
    const uint32_t route = tid + 1024u * i;
    if (route < mineCount) atomicOr(&masks[mine[i] * kWords + route / 32u], 1u << (route % 32u));
  }
  __syncthreads();
  if (tid < p.experts) {
    uint32_t run = 0;
    for (uint32_t w = 0; w < kWords; ++w) {
      before[tid * kWords + w] = uint16_t(run);
      run += uint32_t(__builtin_popcount(masks[tid * kWords + w]));
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t i = 0; i < kMine; ++i) {
    const uint32_t route = tid + 1024u * i;
    if (route >= mineCount) continue;
    const uint32_t at = mine[i] * kWords + route / 32u;
    const uint32_t slot = firstSlot[mine[i]] + before[at] + uint32_t(__builtin_popcount(masks[at] & ((1u << (route % 32u)) - 1u)));
    route_slot[firstRoute + route] = slot;
    slot_row[slot] = (firstRoute + route) / p.top_k;
  }
}
SP_REGISTER_KERNEL("moe_chunk_place", &moe_chunk_place);

// moe_gather_table: the activation table (abi/Gguf.h) of each tile's gathered rows, as
// gguf_prepare_table writes a block's; empty slots are zero rows.
__global__ __launch_bounds__(64) void moe_gather_table(const uint16_t *__restrict__ input, const uint32_t *__restrict__ slot_row,
                                                       const uint32_t *__restrict__ tile_total, uint8_t *__restrict__ tables,
                                                       MoeGatherParams p) {
  const uint32_t g = blockIdx.x, tile = blockIdx.y, lane = threadIdx.x, r = lane & 15u, kq = lane >> 4;
  if (tile >= tile_total[0]) return;
  const uint32_t row = slot_row[tile * MOE_TILE_ROWS + r];
  uint8_t *table = tables + tile * p.table_bytes;
  float v[8];
  uint32_t bits[8] = {};
#pragma unroll
  for (uint32_t e = 0; e < 8; ++e) v[e] = 0.f;
  if (row != MOE_NO_ROW) {
    const uint16_t *x = input + size_t(row) * p.hidden + 32u * g;
#pragma unroll
    for (uint32_t e = 0; e < 8; ++e) {
      bits[e] = x[gguf_operand_input(kq, e)];
      v[e] = bf16_bits_to_float(bits[e]);
    }
  }
  reinterpret_cast<uint4 *>(table)[size_t(g) * 64u + lane] =
      make_uint4(bits[0] | (bits[1] << 16), bits[2] | (bits[3] << 16), bits[4] | (bits[5] << 16), bits[6] | (bits[7] << 16));
  const float half0 = (v[0] + v[2]) + (v[1] + v[3]), half1 = (v[4] + v[6]) + (v[5] + v[7]);
  // (of quarter 0's lanes, the only ones that store them)
  const float s0 = quarters_sum(half0), s1 = quarters_sum(half1);
  if (kq == 0) {
    float *sums32 = reinterpret_cast<float *>(table + gguf_table_sums32_offset(p.hidden, 1));
    float *sums16 = reinterpret_cast<float *>(table + gguf_table_sums16_offset(p.hidden, 1));
    sums32[size_t(g) * 16u + r] = s0 + s1;
    sums16[(2u * size_t(g)) * 16u + r] = s0;
    sums16[(2u * size_t(g) + 1u) * 16u + r] = s1;
  }
}
SP_REGISTER_KERNEL("moe_gather_table", &moe_gather_table);

// moe_combine (moe.metal:367-392): out = bf16(residual + sum over the row's routes of w y) in rank order, fp32.
__global__ __launch_bounds__(256) void moe_combine(const uint16_t *__restrict__ expert_output, const uint32_t *__restrict__ route_slot,
                                                   const float *__restrict__ weights, const uint16_t *__restrict__ residual,
                                                   uint16_t *__restrict__ output, const uint16_t *__restrict__ norm_weight,
                                                   uint8_t *__restrict__ table, MoeCombineParams p) {
  const uint32_t row = blockIdx.x, d = blockIdx.y * 256u + threadIdx.x;
  const bool live = d < p.hidden;  // always, where a table is written
  uint32_t bits = 0;
  if (live) {
    float value = bf16_bits_to_float(residual[size_t(row) * p.hidden + d]);
    // (eight routes' outputs are on their way together; one past the last reads the last and adds nothing)
    constexpr uint32_t kAhead = 8;
    for (uint32_t first = 0; first < p.top_k; first += kAhead) {
      float weight[kAhead];
      uint32_t y[kAhead];
#pragma unroll
      for (uint32_t i = 0; i < kAhead; ++i) {
        const size_t route = size_t(row) * p.top_k + min(first + i, p.top_k - 1u);
        weight[i] = weights[route];
        y[i] = expert_output[size_t(route_slot[route]) * p.hidden + d];
      }
#pragma unroll
      for (uint32_t i = 0; i < kAhead; ++i)
        if (first + i < p.top_k) value += weight[i] * bf16_bits_to_float(y[i]);
    }
    bits = float_to_bf16_bits(value);
    output[size_t(row) * p.hidden + d] = uint16_t(bits);
  }
  if (!p.table_tiles) return;
  // The row's piece of the table: lane l of a wave holds input 64 j + l of column group j. Runs of four
  // inputs are one 8-byte piece of a table entry; lanes 4 i lead them.
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, r = row % 16u, G = p.hidden / 32u;
  const uint32_t piece = row / 16u / GGUF_PIECE_TILES, tile = row / 16u % GGUF_PIECE_TILES;
  const uint32_t tiles = min(uint32_t(GGUF_PIECE_TILES), p.table_tiles - piece * GGUF_PIECE_TILES);
  table += piece * gguf_table_bytes(p.hidden, GGUF_PIECE_TILES);
  const float hidden = bf16_bits_to_float(bits);
  const uint32_t scaled = float_to_bf16_bits(hidden * bf16_bits_to_float(norm_weight[d]));
  const float v = bf16_bits_to_float(scaled);
  const uint32_t b1 = lane_down<1>(scaled), b2 = lane_down<2>(scaled), b3 = lane_down<3>(scaled);
  const float v1 = lane_down<1>(v), v2 = lane_down<2>(v), v3 = lane_down<3>(v);
  // sums of 16 inputs in input order: the four runs of a half are led by lanes 4 apart
  float s = (v + v1) + (v2 + v3);
  const float s1 = lane_down<4>(s), s2 = lane_down<8>(s), s3 = lane_down<12>(s);
  s = ((s + s1) + s2) + s3;
  const float other = lane_xor<16>(s);
  float square = hidden * hidden;
  square = row_sum_dpp(square);
  square += lane_xor<16>(square);
  square += lane_xor<32>(square);
  const uint32_t q = d / 4u, g = q / 8u, half = (q / 4u) % 2u, kq = q % 4u;  // the run of input d
  if ((lane & 3u) == 0) {
    // operand elements 4 half + {0,1,2,3} are inputs 4 kq + {0,2,1,3} of the half
    reinterpret_cast<uint2 *>(table)[((size_t(tile) * G + g) * 64u + kq * 16u + r) * 2u + half] =
        make_uint2(scaled | (b2 << 16), b1 | (b3 << 16));
    if (kq == 0) {
      float *sums32 = reinterpret_cast<float *>(table + gguf_table_sums32_offset(p.hidden, tiles));
      float *sums16 = reinterpret_cast<float *>(table + gguf_table_sums16_offset(p.hidden, tiles));
      sums16[(size_t(tile) * 2u * G + 2u * g + half) * 16u + r] = s;
      if (half == 0) sums32[(size_t(tile) * G + g) * 16u + r] = s + other;
    }
  }
  if (lane == 0) {
    float *squares = reinterpret_cast<float *>(table + gguf_table_squares_offset(p.hidden, tiles));
    squares[size_t(blockIdx.y * 4u + wave) * gguf_squares_stride(tiles) + 16u * tile + r] = square;
  }
}
SP_REGISTER_KERNEL("moe_combine", &moe_combine);

// moe_combine_rows: the same rows without a table, grid (rows, ceil(hidden / 2048)), 256 threads, eight columns a thread by
// 16-byte loads (the buffers' alignment is the host's rule), eight routes' loads out together. 2048 rows of 2048 columns
// and 8 routes: a column a thread 31 us (2.7 TB/s), eight 14.
__global__ __launch_bounds__(256) void moe_combine_rows(const uint16_t *__restrict__ expert_output, const uint32_t *__restrict__ route_slot,
                                                        const float *__restrict__ weights, const uint16_t *__restrict__ residual,
                                                        uint16_t *__restrict__ output, MoeCombineParams p) {
  constexpr uint32_t kTogether = 8u;
  const uint32_t row = blockIdx.x, d = (blockIdx.y * 256u + threadIdx.x) * 8u;
  if (d >= p.hidden) return;
  auto widen = [](const uint4 &v, float (&to)[8]) __attribute__((always_inline)) {
    const uint32_t words[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      to[2 * i] = bf16_bits_to_float(words[i] & 0xFFFFu);
      to[2 * i + 1] = bf16_bits_to_float(words[i] >> 16);
    }
  };
  float value[8];
  widen(*reinterpret_cast<const uint4 *>(residual + size_t(row) * p.hidden + d), value);
  for (uint32_t rank0 = 0; rank0 < p.top_k; rank0 += kTogether) {
    uint4 rows[kTogether];
    float weight[kTogether];
#pragma unroll
    for (uint32_t i = 0; i < kTogether; ++i) {
      const size_t route = size_t(row) * p.top_k + min(rank0 + i, p.top_k - 1u);   // the last route again past the row's
      weight[i] = weights[route];
      rows[i] = *reinterpret_cast<const uint4 *>(expert_output + size_t(route_slot[route]) * p.hidden + d);
    }
#pragma unroll
    for (uint32_t i = 0; i < kTogether; ++i) {
      if (rank0 + i >= p.top_k) break;
      float y[8];
      widen(rows[i], y);
#pragma unroll
      for (int c = 0; c < 8; ++c) value[c] += weight[i] * y[c];
    }
  }
  uint32_t bits[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) bits[c] = float_to_bf16_bits(value[c]);
  *reinterpret_cast<uint4 *>(output + size_t(row) * p.hidden + d) =
      make_uint4(bits[0] | (bits[1] << 16), bits[2] | (bits[3] << 16), bits[4] | (bits[5] << 16), bits[6] | (bits[7] << 16));
}
SP_REGISTER_KERNEL("moe_combine_rows", &moe_combine_rows);

} // namespace splash::kernels
