// Acceptance of a verify block (the reference's kernels/decode/sampling.metal: argmax_shard
// :1896-1961, argmax_reduce :1963-1997, shard_mass / merge_masses :102-154, vocabulary_draw
// :713-885, decode_accept_tree :2044-2083), on 64-lane wavefronts.
//
// Greedy rows: SAMPLING_SHARDS workgroups scan a row's logits, each thread its tokens in id order
// (shard * 256 + tid + n * shards * 256), keeping the larger value and, among equals, the lower id;
// NaN and -inf are never selected; the shards' partials reduce by the same rule. A row with no
// selectable logit selects SAMPLING_NO_TOKEN.
//
// Sampled rows (temperature > 0): weight_t = exp((logit_t - max) / T). One pass gives each shard's
// online (max, sum), merged in shard order. The row's drafted child d is accepted iff
// u_child * q_d < p_d, p = weight / total. Otherwise the row draws from the residual
// max(p - q, 0): SAMPLING_RANGES id-ordered ranges are summed (a thread sums its chunk of a range in
// id order, the chunks are added in order), the ranges are walked in order to the one that holds
// point = u_row * sum, then its chunks and the hit chunk's tokens, each in id order; rounding
// fall-backs take the last weighted range, chunk and token. A row without a child draws the same
// way from p itself.
//
// A lane's min_p, top_k and top_p cut its rows' distributions (distribution_end, sampling.metal:
// 603-670): in the order of the logits (larger first, among equals the smaller id first) a row keeps
// the tokens at or above the logit that weighs min_p of the heaviest, then the first top_k of those,
// then of those the tokens up to the one at which their mass first exceeds top_p of the kept mass.
// The end is found by radix descent over the order-preserving key of a logit, four bits a pass, each
// pass one scan of the row with a 16-bin histogram of counts and masses (a thread's tokens in id
// order, the threads' sums in a fixed tree), then over the ids of the tokens tied at the last key.
// Everything after it weighs nothing; p is renormalized by the kept mass.
#include "abi/Sampling.h"
#include "abi/PagedAttention.h"
#include "backend/KernelRegistry.hpp"
#include "kernels/acceptance.hpp"

#include <cfloat>

namespace splash::kernels {

__device__ __forceinline__ uint32_t lane_of(const TargetSamplingParams &p, uint32_t row) {
  uint32_t lane = 0;
  for (uint32_t l = 0; l < p.lanes; ++l)
    if (row >= p.lane[l].first && row < p.lane[l].first + p.lane[l].rows) lane = l;
  return lane;
}
// decode_sample_admit: grid (rows, ceil(vocabulary / 1024)), 256 threads. A row of a constrained lane
// admits only the tokens of its constraint-mask row, a row of a lane that ignores end-of-sequence no
// stop token (TargetRow::admits, sampling.metal:42-46): the logits of the others become -infinity,
// which every selection kernel leaves out, before any of them reads the row.
__global__ __launch_bounds__(256) void decode_sample_admit(float *__restrict__ logits, const uint32_t *__restrict__ token_mask,
                                                           TargetSamplingParams p) {
  const uint32_t row = blockIdx.x, lane = lane_of(p, row);
  const bool constrained = (p.constrained_mask >> lane) & 1u, excludes = (p.exclude_stop_mask >> lane) & 1u;
  if (!constrained && !excludes) return;
  float *x = logits + size_t(row) * p.logits_stride;
  const uint32_t *mask = token_mask + size_t(row) * p.mask_words;
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    const uint32_t token = (blockIdx.y * 4u + i) * 256u + threadIdx.x;
    if (token >= p.vocabulary) continue;
    bool admitted = !constrained || ((mask[token / 32u] >> (token % 32u)) & 1u);
    if (excludes)
      for (uint32_t s = 0; s < SAMPLING_STOP_TOKENS; ++s) admitted = admitted && token != p.stop_tokens[s];
    if (!admitted) x[token] = -INFINITY;
  }
}
SP_REGISTER_KERNEL("decode_sample_admit", &decode_sample_admit);

// The sampling penalties of one logit (PenaltyReference.hpp:27-40, sampling.metal:991-1006 in the reference): the
// repetition penalty divides a positive logit and multiplies another when the prompt or the output holds the token;
// presence and frequency lower it by the output's count of the token; the result stays finite. NaN and -infinity, which
// no selection takes, stay as they are. One product, one product and sum, one difference, each rounded once.
__device__ __forceinline__ float penalized_logit(float value, uint32_t count, float repetition, float repetition_inverse, float presence,
                                                 float frequency) {
  const uint32_t bits = __float_as_uint(value);
  if ((bits & 0x7FFFFFFFu) > 0x7F800000u || bits == 0xFF800000u) return value;
  float v = value * (value > 0.0f ? repetition_inverse : repetition);
  if (count) v = v - (frequency * float(count) + presence);
  return fminf(fmaxf(v, -3.402823466e+38f), 3.402823466e+38f);
}
// decode_sample_penalize: grid (ceil(vocabulary / 1024), entries), 256 threads, four tokens a thread 256 apart. A token
// that the entry's table row does not hold and no row of the block drafted is left alone (nearly every token). A row's
// context adds, to the table's count, the block's draft tokens on its path: its ancestors' and its own input token, but
// not the anchor's, which the table counted when the target selected it (sampling.metal:1008-1050).
__global__ __launch_bounds__(256) void decode_sample_penalize(float *__restrict__ logits, const uint32_t *__restrict__ words,
                                                              const uint32_t *__restrict__ input_tokens,
                                                              const AttentionTreeRow *__restrict__ tree, SamplingPenaltyParams p) {
  const uint32_t entry = blockIdx.y;
  const SamplingLaneRows lane = p.lane[entry];
  __shared__ uint32_t drafts[SAMPLING_MAXIMUM_ROWS], paths[SAMPLING_MAXIMUM_ROWS];
  if (threadIdx.x < lane.rows) {
    drafts[threadIdx.x] = input_tokens[lane.first + threadIdx.x];
    paths[threadIdx.x] = tree[lane.first + threadIdx.x].ancestors & ~1u;
  }
  __syncthreads();
  const float repetition = p.repetition[entry], inverse = p.repetition_inverse[entry], presence = p.presence[entry],
              frequency = p.frequency[entry];
  const uint32_t *row_words = words + size_t(p.table_row[entry]) * p.vocabulary;
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    const uint32_t token = (blockIdx.x * 4u + i) * 256u + threadIdx.x;
    if (token >= p.vocabulary) continue;
    const uint32_t word = row_words[token];
    uint32_t drafted = 0;
    for (uint32_t r = 1; r < lane.rows; ++r) drafted |= uint32_t(drafts[r] == token) << r;
    if (!(word | drafted)) continue;
    const uint32_t selected = word & SAMPLING_PENALTY_COUNT;
    float *column = logits + size_t(lane.first) * p.logits_stride + token;
    for (uint32_t r = 0; r < lane.rows; ++r) {
      const uint32_t count = selected + uint32_t(__popc(drafted & paths[r]));
      if (!count && !(word & SAMPLING_PENALTY_PROMPT)) continue;
      float &x = column[size_t(r) * p.logits_stride];
      x = penalized_logit(x, count, repetition, inverse, presence, frequency);
    }
  }
}
SP_REGISTER_KERNEL("decode_sample_penalize", &decode_sample_penalize);

// decode_sample_count_tokens: grid (entries), 64 threads. The tokens a lane retained of a step (the acceptance's `tokens`
// from the lane's first row, `retained` of them) are counted into its row of the penalty table on the device, where the
// reference's engine counts them on the host into shared memory (Sampling::countPenaltyTokens, Sampling.cpp:116-121).
// A token twice in one step is counted twice (atomic adds).
__global__ __launch_bounds__(64) void decode_sample_count_tokens(uint32_t *__restrict__ words, const uint32_t *__restrict__ tokens,
                                                                 const uint32_t *__restrict__ retained, SamplingCountParams p) {
  const uint32_t entry = blockIdx.x;
  const uint32_t count = min(retained[p.lane[entry]], uint32_t(SAMPLING_MAXIMUM_ROWS));
  if (threadIdx.x >= count) return;
  const uint32_t token = tokens[p.first_row[entry] + threadIdx.x];
  if (token < p.vocabulary) atomicAdd(words + size_t(p.table_row[entry]) * p.vocabulary + token, 1u);
}
SP_REGISTER_KERNEL("decode_sample_count_tokens", &decode_sample_count_tokens);

// decode_sample_end_thinking: grid (lanes), 64 threads, a thread a row of the lane's block (the reference walks a lane's
// rows in one thread, sampling.metal:1993-2039; every row reads and writes its own selection only, so they go side by
// side). The k-th row of a path, ascending, is its row of depth k.
__global__ __launch_bounds__(64) void decode_sample_end_thinking(const uint32_t *__restrict__ input_tokens,
                                                                 const uint32_t *__restrict__ token_mask,
                                                                 const AttentionTreeRow *__restrict__ tree, uint32_t *__restrict__ tokens,
                                                                 ThinkingCutoffParams p) {
  const uint32_t lane = blockIdx.x;
  const SamplingLaneRows block = p.lane[lane];
  if (threadIdx.x >= block.rows || p.row[lane] >= SAMPLING_MAXIMUM_ROWS) return;
  const uint32_t mine = block.first + threadIdx.x;
  const uint32_t path = tree[mine].ancestors, depth = tree[mine].depth;
  const bool waits = (p.waiting_mask >> lane) & 1u;
  const uint32_t start = p.tokens[lane][0];
  // the cut: the first depth from the lane's row on (whose row admits the end's first token, where the end waits)
  uint32_t cut = 0, left = path;
  bool found = false;
  for (; left; left &= left - 1u, ++cut) {
    if (cut < p.row[lane]) continue;
    const uint32_t at = block.first + uint32_t(__ffs(int(left)) - 1);
    if (!waits || ((token_mask[size_t(at) * p.mask_words + start / 32u] >> (start % 32u)) & 1u)) {
      found = true;
      break;
    }
  }
  if (!found || cut > depth || depth - cut >= p.count[lane]) return;
  // thinking that a draft token ended at or before the cut stays ended
  for (uint32_t before = path & ~1u; before; before &= before - 1u) {
    const uint32_t at = block.first + uint32_t(__ffs(int(before)) - 1);
    const uint32_t draft = input_tokens[at];
    if (tree[at].depth <= cut && (draft == p.close[lane] || draft == p.also_ends[lane])) return;
  }
  if (tokens[mine] < p.vocabulary) tokens[mine] = p.tokens[lane][depth - cut];
}
SP_REGISTER_KERNEL("decode_sample_end_thinking", &decode_sample_end_thinking);


// draft_verify_rows (the layout the reference's sampling.metal:1799-1895 produces): lane l's tree holds sizes[l] rows
// from row l * 16 of tree_tokens, trees and scores (a row's draft probability and its estimate, the chance that the
// target accepts it), in the order the selector took them, best first. The step takes every lane's anchor and the
// best other rows by estimate (among equals the lower lane, then the lower row) that its rows and the lanes' cap
// hold, none below the floor; a lane's rows are numbered in preorder, the earlier-taken child first, so that the
// likeliest path of its tree lies on its first rows; the rows of no lane carry lane 0's anchor, no path and no source.
//
// One workgroup of 128 threads, thread (lane, row) = (t / 16, t % 16), no loop over the step's rows:
//   rank      a candidate's place in the order above is the count of candidates that beat it;
//   take      in that order a candidate is eligible if it is at or above the floor and fewer than cap - 1 candidates
//             of its lane precede it; it is taken if fewer than rows - lanes eligible ones precede it (wave ballots
//             over the ranked order);
//   preorder  with ancestor masks, row x precedes row r if x is an ancestor of r or, where their paths part, x's
//             branch was taken earlier (parents are taken before children, so the lowest set bit of a path below
//             the common part is its branch): r's place is the count of the lane's rows that precede it.
__global__ __launch_bounds__(128) void draft_verify_rows(const uint32_t *__restrict__ tree_tokens, const AttentionTreeRow *__restrict__ trees,
                                                         const float2 *__restrict__ scores, const uint32_t *__restrict__ sizes,
                                                         uint32_t *__restrict__ tokens, AttentionTreeRow *__restrict__ tree,
                                                         SamplingLaneRows *__restrict__ lane_rows, uint32_t *__restrict__ sources,
                                                         VerifyRowsParams p) {
  constexpr uint32_t kLanes = SAMPLING_MAXIMUM_LANES, kRows = SAMPLING_MAXIMUM_ROWS, kAll = kLanes * kRows;
  __shared__ __align__(16) float estimateOf[kAll];
  __shared__ uint32_t rankedOwner[kAll];   // the lane of the candidate at each place of the order, kLanes for none
  __shared__ float rankedEstimate[kAll];
  __shared__ uint32_t eligibleBefore[2];   // eligible candidates in the first wave's places
  __shared__ __align__(16) uint32_t takenOf[kLanes];
  __shared__ __align__(16) uint32_t pathOf[kAll];   // a row's ancestors and itself, in its tree's own numbering
  __shared__ __align__(16) uint32_t placeOf[kAll];  // a row's place in its lane's preorder
  // (the lists are read whole, sixteen bytes at a time, before the first of them is used: entry by entry each would be waited for)
  auto four = [](const uint32_t *from, uint32_t i, uint32_t (&to)[4]) {
    const uint4 v = reinterpret_cast<const uint4 *>(from)[i];
    to[0] = v.x, to[1] = v.y, to[2] = v.z, to[3] = v.w;
  };
  if (blockIdx.x) return;
  const uint32_t t = threadIdx.x, lane = t / kRows, row = t % kRows, lanes = min(p.lanes, kLanes);
  const uint32_t size = lane < lanes ? min(sizes[lane], kRows) : 0u;
  const bool candidate = row >= 1 && row < size;
  // (all that is read of a row is on its way at once: the kernel is one workgroup's chain of waits)
  const bool held = lane < lanes;
  const float scored = held ? scores[t].y : 0.f;
  const AttentionTreeRow read = held ? trees[t] : AttentionTreeRow{0u, 0u, 0u};
  const uint32_t token = held ? tree_tokens[t] : 0u;
  const float estimate = candidate ? scored : 0.f;
  estimateOf[t] = candidate ? estimate : -INFINITY;
  rankedOwner[t] = kLanes;
  rankedEstimate[t] = -INFINITY;
  if (t < kLanes) takenOf[t] = 0;
  __syncthreads();
  if (candidate) {
    uint32_t rank = 0;
#pragma unroll
    for (uint32_t i = 0; i < kAll / 4u; ++i) {   // (no candidate: -infinity)
      const float4 e4 = reinterpret_cast<const float4 *>(estimateOf)[i];
      const float e[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) rank += (e[k] > estimate || (e[k] == estimate && 4u * i + k < t)) && e[k] != -INFINITY ? 1u : 0u;
    }
    rankedOwner[rank] = lane;
    rankedEstimate[rank] = estimate;
  }
  __syncthreads();
  // Thread t now stands for place t of the order.
  const uint32_t owner = rankedOwner[t];
  uint32_t before = 0;   // candidates of the same lane at earlier places
  const uint64_t earlierLanes = (uint64_t{1} << (t & 63u)) - 1u;
  const uint32_t firstOwner = rankedOwner[t & 63u];   // (the first wave's places, for the second)
#pragma unroll
  for (uint32_t l = 0; l < kLanes; ++l) {
    const uint64_t here = __builtin_amdgcn_ballot_w64(owner == l), ahead = __builtin_amdgcn_ballot_w64(t >= 64u && firstOwner == l);
    if (owner == l) before = uint32_t(__builtin_popcountll(here & earlierLanes) + __builtin_popcountll(ahead));
  }
  const bool eligible = owner < kLanes && !(rankedEstimate[t] < p.floor) && before + 1u < p.lane_cap;
  const uint64_t ballot = __builtin_amdgcn_ballot_w64(eligible);
  if ((t & 63u) == 0) eligibleBefore[t >> 6] = uint32_t(__builtin_popcountll(ballot));
  __syncthreads();
  const uint32_t earlier = uint32_t(__builtin_popcountll(ballot & earlierLanes)) + (t >= 64 ? eligibleBefore[0] : 0u);
  const uint32_t budget = p.rows > lanes ? p.rows - lanes : 0u;
  if (eligible && earlier < budget) atomicAdd(&takenOf[owner], 1u);
  __syncthreads();
  // Back to thread (lane, row): the lane keeps its anchor and its first taken rows.
  uint32_t mine = 0, first = 0, total = 0;
#pragma unroll
  for (uint32_t i = 0; i < kLanes / 4u; ++i) {
    uint32_t taken[4];
    four(takenOf, i, taken);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      const uint32_t l = 4u * i + k, here = l < lanes ? taken[k] + 1u : 0u;
      mine = l == lane ? here : mine;
      first += l < lane ? here : 0u;
      total += here;
    }
  }
  if (p.slots) first = lane * p.lane_cap;
  const bool placed = row < mine;
  const AttentionTreeRow node = placed ? read : AttentionTreeRow{0u, 0u, 0u};
  pathOf[t] = placed ? node.ancestors : 0u;
  __syncthreads();
  static_assert(kRows == 16 && kLanes % 4 == 0, "a lane's rows are four reads");
  uint32_t place = 0;
  if (placed) {
    const uint32_t path = node.ancestors;
#pragma unroll
    for (uint32_t i = 0; i < kRows / 4u; ++i) {
      uint32_t paths[4];
      four(pathOf + lane * kRows, i, paths);
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t x = 4u * i + k, other = paths[k], common = other & path;
        const bool ancestor = (path >> x) & 1u, descendant = (other >> row) & 1u;
        const bool earlierBranch = __builtin_ctz((other & ~common) | 0x10000u) < __builtin_ctz((path & ~common) | 0x10000u);
        place += x < mine && x != row && (ancestor || (!descendant && earlierBranch)) ? 1u : 0u;
      }
    }
  }
  placeOf[t] = place;
  __syncthreads();
  if (placed) {
    uint32_t ancestors = 0;
#pragma unroll
    for (uint32_t i = 0; i < kRows / 4u; ++i) {
      uint32_t places[4];
      four(placeOf + lane * kRows, i, places);
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) ancestors |= (node.ancestors >> (4u * i + k) & 1u) << (places[k] & 31u);
    }
    const uint32_t depth = uint32_t(__builtin_popcount(node.ancestors)) - 1u;
    const uint32_t up = row ? placeOf[lane * kRows + node.parent] : SAMPLING_TREE_ROOT;
    tokens[first + place] = token;
    tree[first + place] = AttentionTreeRow{ancestors, uint16_t(up), uint16_t(depth)};
    sources[first + place] = row;
  }
  if (lane < lanes && row == 0) lane_rows[lane] = SamplingLaneRows{first, mine};
  if (p.slots) {
    // the rows of a lane's slot past its own: inert
    if (lane < lanes && row >= mine && row < p.lane_cap) {
      tokens[first + row] = SAMPLING_NO_TOKEN;
      tree[first + row] = AttentionTreeRow{1u << row, uint16_t(0), uint16_t(1)};
      sources[first + row] = SAMPLING_NO_TOKEN;
    }
    return;
  }
  for (uint32_t spare = total + t; spare < p.rows; spare += kAll) {
    tokens[spare] = tree_tokens[0];
    tree[spare] = AttentionTreeRow{0u, uint16_t(SAMPLING_TREE_ROOT), uint16_t(0)};
    sources[spare] = SAMPLING_NO_TOKEN;
  }
}
SP_REGISTER_KERNEL("draft_verify_rows", &draft_verify_rows);

// A thread's tokens of a shard, in id order: every SAMPLING_SHARDS * 256th from its own. Their loads are on their way eight
// together (one past the vocabulary reads the last and is not taken); one at a time each waited for the one before: 16 rows
// of 151936 logits 10 us, 6 so.
template <class Take> __device__ __forceinline__ void shard_scan(const float *x, uint32_t vocabulary, uint32_t shard, uint32_t tid, Take take) {
  constexpr uint32_t kAhead = 8, kStep = SAMPLING_SHARDS * 256u;
  for (uint32_t first = shard * 256u + tid; first < vocabulary; first += kAhead * kStep) {
    float values[kAhead];
#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i) values[i] = __builtin_nontemporal_load(x + min(first + i * kStep, vocabulary - 1u));
#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i)
      if (first + i * kStep < vocabulary) take(values[i], first + i * kStep);
  }
}

// Grid (rows * SAMPLING_SHARDS), 256 threads. partial_values/indices [row][shard].
__global__ __launch_bounds__(256) void decode_sample_argmax_sharded(const float *__restrict__ logits, float *__restrict__ partial_values,
                                                                    uint32_t *__restrict__ partial_indices, TargetSamplingParams p) {
  __shared__ float values[4];
  __shared__ uint32_t indices[4];
  const uint32_t row = blockIdx.x / SAMPLING_SHARDS, shard = blockIdx.x % SAMPLING_SHARDS, tid = threadIdx.x;
  const float *x = logits + size_t(row) * p.logits_stride;
  Best best{-INFINITY, SAMPLING_NO_TOKEN};
  shard_scan(x, p.vocabulary, shard, tid, [&](float value, uint32_t token) {
    if (!unselectable(value) && (value > best.value || (value == best.value && token < best.index))) best = {value, token};
  });
  best = wave_best(best);
  if ((tid & 63u) == 0) {
    values[tid >> 6] = best.value;
    indices[tid >> 6] = best.index;
  }
  __syncthreads();
  if (tid == 0) {
    Best all{values[0], indices[0]};
#pragma unroll
    for (int w = 1; w < 4; ++w) all = better(all, Best{values[w], indices[w]});
    partial_values[blockIdx.x] = all.value;
    partial_indices[blockIdx.x] = all.index;
  }
}
SP_REGISTER_KERNEL("decode_sample_argmax_sharded", &decode_sample_argmax_sharded);

// Grid (rows), 64 threads: the row's token from its shards' partials.
__global__ __launch_bounds__(64) void decode_sample_argmax_reduce(const float *__restrict__ partial_values,
                                                                  const uint32_t *__restrict__ partial_indices,
                                                                  uint32_t *__restrict__ tokens, TargetSamplingParams p) {
  const uint32_t row = blockIdx.x, tid = threadIdx.x;
  Best best{-INFINITY, SAMPLING_NO_TOKEN};
  if (tid < SAMPLING_SHARDS) best = {partial_values[row * SAMPLING_SHARDS + tid], partial_indices[row * SAMPLING_SHARDS + tid]};
  if (unselectable(best.value)) best = {-INFINITY, SAMPLING_NO_TOKEN};
  best = wave_best(best);
  if (tid == 0) tokens[row] = best.index;
}
SP_REGISTER_KERNEL("decode_sample_argmax_reduce", &decode_sample_argmax_reduce);

// decode_accept_tree (what the reference's sampling.metal:2044-2083 decides): grid (lanes), one wavefront a lane, a
// thread a row (accept_rows). tokens: in, each row's selection; out, the lane's retained tokens from its first row.
__global__ __launch_bounds__(64) void decode_accept_tree(const uint32_t *__restrict__ input_tokens, const AttentionTreeRow *__restrict__ tree,
                                                         uint32_t *__restrict__ tokens, uint32_t *__restrict__ retained,
                                                         uint32_t *__restrict__ accepted_count, uint32_t *__restrict__ retained_rows,
                                                         AcceptBatchParams p) {
  const uint32_t lane = blockIdx.x, row = threadIdx.x;
  if (lane >= p.lanes) return;
  const uint32_t first = p.lane[lane].first, rows = min(p.lane[lane].rows, SAMPLING_MAXIMUM_ROWS);
  const bool live = row < rows;
  const AttentionTreeRow node = live ? tree[first + row] : AttentionTreeRow{0u, 0u, 0u};
  const uint32_t input = live ? input_tokens[first + row] : 0u, selection = live ? tokens[first + row] : 0u;
  const Acceptance a = accept_rows(row, live, node, input, selection, p.remaining[lane], p.stop_tokens);
  if (a.retains) tokens[first + a.depth] = selection;   // every selection was read before any is written
  if (a.last) {
    retained_rows[lane] = node.ancestors;
    retained[lane] = a.kept;
    accepted_count[lane] = a.accepted;
  }
}
SP_REGISTER_KERNEL("decode_accept_tree", &decode_accept_tree);

// ---------------------------------------------------------------------------------------------
// Sampled rows.
// ---------------------------------------------------------------------------------------------
struct Mass {
  float maximum, sum;
};
// merge_masses (sampling.metal:122-154): the larger maximum first, then both sums at it.
__device__ __forceinline__ Mass merge(Mass a, Mass b, float inverse_temperature) {
  const float m = fmaxf(a.maximum, b.maximum);
  if (m == -INFINITY) return {m, 0.f};
  // the side that holds the maximum weighs exp(0) = 1: one exponential, of the other side
  const bool first = a.maximum == m;
  const float other = (first ? b.maximum : a.maximum), weight = other == -INFINITY ? 0.f : expf((other - m) * inverse_temperature);
  const float sa = first ? a.sum : a.sum * weight, sb = first ? b.sum * weight : b.sum;
  return {m, sa + sb};
}
__device__ __forceinline__ uint32_t lane_of_row(const TargetSamplingParams &p, uint32_t row) {
  uint32_t lane = 0;
  for (uint32_t l = 0; l < p.lanes; ++l)
    if (row >= p.lane[l].first && row < p.lane[l].first + p.lane[l].rows) lane = l;
  return lane;
}

// Grid (rows * SAMPLING_SHARDS), 256 threads: the shard's online (max, sum). masses [row][shard][2].
__global__ __launch_bounds__(256) void decode_sample_mass_sharded(const float *__restrict__ logits, float *__restrict__ masses,
                                                                  TargetSamplingParams p) {
  __shared__ float shared[4][2];
  const uint32_t row = blockIdx.x / SAMPLING_SHARDS, shard = blockIdx.x % SAMPLING_SHARDS, tid = threadIdx.x;
  const float inverse = 1.0f / p.temperature[lane_of_row(p, row)];
  const float *x = logits + size_t(row) * p.logits_stride;
  Mass mine{-INFINITY, 0.f};
  shard_scan(x, p.vocabulary, shard, tid, [&](float value, uint32_t) {
    if (!unselectable(value)) mine = merge(mine, Mass{value, 1.0f}, inverse);
  });
  // lanes in a fixed butterfly, then the four wavefronts in order
  mine = merge(mine, Mass{lane_xor<32>(mine.maximum), lane_xor<32>(mine.sum)}, inverse);
  mine = merge(mine, Mass{lane_xor<16>(mine.maximum), lane_xor<16>(mine.sum)}, inverse);
  mine = merge(mine, Mass{lane_xor<8>(mine.maximum), lane_xor<8>(mine.sum)}, inverse);
  mine = merge(mine, Mass{lane_xor<4>(mine.maximum), lane_xor<4>(mine.sum)}, inverse);
  mine = merge(mine, Mass{lane_xor<2>(mine.maximum), lane_xor<2>(mine.sum)}, inverse);
  mine = merge(mine, Mass{lane_xor<1>(mine.maximum), lane_xor<1>(mine.sum)}, inverse);
  if ((tid & 63u) == 0) {
    shared[tid >> 6][0] = mine.maximum;
    shared[tid >> 6][1] = mine.sum;
  }
  __syncthreads();
  if (tid == 0) {
    Mass all{shared[0][0], shared[0][1]};
#pragma unroll
    for (int w = 1; w < 4; ++w) all = merge(all, Mass{shared[w][0], shared[w][1]}, inverse);
    masses[2 * blockIdx.x] = all.maximum;
    masses[2 * blockIdx.x + 1] = all.sum;
  }
}
SP_REGISTER_KERNEL("decode_sample_mass_sharded", &decode_sample_mass_sharded);

// The row's (max, total) from its shards: every shard's sum at the row's maximum, a lane a shard, added in shard order.
// Called by whole wavefronts. (Merged one after the other, an exponential each waiting for the last, they took 4 us of every
// kernel that asks.)
__device__ __forceinline__ Mass row_mass(const float *masses, uint32_t row, float inverse) {
  const uint32_t shard = (threadIdx.x & 63u) % SAMPLING_SHARDS;
  const float2 mine = reinterpret_cast<const float2 *>(masses)[row * SAMPLING_SHARDS + shard];
  const float maximum = wave_max(mine.x);
  // (a shard at the maximum weighs 1 as it is: of an infinite maximum, or divided by the least temperatures, 0 is no number)
  const float sum = mine.x == maximum ? mine.y : mine.x == -INFINITY ? 0.f : mine.y * expf((mine.x - maximum) * inverse);
  float total = 0.f;
#pragma unroll
  for (int s = 0; s < int(SAMPLING_SHARDS); ++s) total += lane_value_of(sum, s);
  return {maximum, total};
}
// The child of `row` in its lane's block: the first later row whose parent it is; none: SAMPLING_NO_TOKEN.
__device__ __forceinline__ uint32_t child_token(const TargetSamplingParams &p, const AttentionTreeRow *tree,
                                                const uint32_t *input_tokens, uint32_t row) {
  const uint32_t lane = lane_of_row(p, row), first = p.lane[lane].first, local = row - first;
  for (uint32_t child = local + 1; child < p.lane[lane].rows; ++child)
    if (tree[first + child].parent == local) return input_tokens[first + child];
  return SAMPLING_NO_TOKEN;
}
// The order of the logits as an unsigned key (sampling.metal:197-207): a larger logit has a larger
// key; -0 and +0 share one; every finite logit's key is above that of -infinity.
__device__ __forceinline__ uint32_t logit_key(float value) {
  uint32_t bits = __builtin_bit_cast(uint32_t, value);
  bits = (bits << 1) ? bits : 0u;
  return (bits & 0x80000000u) ? ~bits : bits | 0x80000000u;
}
__device__ __forceinline__ float key_logit(uint32_t key) {
  return __builtin_bit_cast(float, (key & 0x80000000u) ? key & 0x7FFFFFFFu : ~key);
}
// A position in the order: the tokens at or before it have a larger key, or its key and an id at
// most `last`. {0, 0} lies after every token.
struct OrderEnd {
  uint32_t key, last;
};
__device__ __forceinline__ bool at_or_before(uint32_t key, uint32_t token, OrderEnd end) {
  return key > end.key || (key == end.key && token <= end.last);
}
// A row's distribution: its maximum, the mass of the tokens it keeps and the last of them.
struct Kept {
  Mass mass;  // maximum, kept mass
  OrderEnd end;
};
__device__ __forceinline__ Kept row_kept(const float *masses, const uint32_t *decisions, uint32_t row, float inverse, bool truncating) {
  Kept kept{row_mass(masses, row, inverse), {0u, 0u}};
  if (truncating) {
    const uint32_t *words = decisions + size_t(row) * SAMPLING_DECISION_WORDS;
    kept.end = {words[SAMPLING_END_KEY], words[SAMPLING_END_LAST]};
    kept.mass.sum = __builtin_bit_cast(float, words[SAMPLING_END_MASS]);
  }
  return kept;
}
__device__ __forceinline__ float token_weight(float logit, Mass mass, float inverse) {
  return unselectable(logit) ? 0.f : expf((logit - mass.maximum) * inverse);
}
// A token's weight in the row's distribution: its softmax weight at or before the end, else 0 (kept_weight, sampling.metal:672-679).
__device__ __forceinline__ float kept_weight(float logit, uint32_t token, const Kept &kept, float inverse) {
  if (unselectable(logit) || !at_or_before(logit_key(logit), token, kept.end)) return 0.f;
  return expf((logit - kept.mass.maximum) * inverse);
}
// The residual weight of token t: max(p_t - q_t, 0) after a rejection, p_t's weight otherwise.
__device__ __forceinline__ float residual_of(float logit, uint32_t token, float q, const Kept &kept, float inverse, bool rejected) {
  const float w = kept_weight(logit, token, kept, inverse);
  return rejected ? fmaxf(w / kept.mass.sum - q, 0.f) : w;
}
// The residual weights of tokens first .. first + count, below end, summed in order; eight tokens' loads are on their way
// together (one past the end reads the last and adds nothing).
__device__ __forceinline__ float lane_residual(const float *x, const float *q, uint32_t first, uint32_t count, uint32_t end, const Kept &kept,
                                               float inverse, bool rejected) {
  constexpr uint32_t kAhead = 8;
  float sum = 0.f;
  for (uint32_t i0 = 0; i0 < count; i0 += kAhead) {
    float logits[kAhead], drafted[kAhead];
#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i) {
      const uint32_t at = min(first + i0 + i, end - 1u);
      logits[i] = x[at];
      drafted[i] = rejected ? q[at] : 0.f;
    }
#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i)
      if (i0 + i < count && first + i0 + i < end) sum += residual_of(logits[i], first + i0 + i, drafted[i], kept, inverse, rejected);
  }
  return sum;
}
// ---------------------------------------------------------------------------------------------
// decode_sample_distribution_end: grid (rows), 1024 threads. Writes the row's end words of the
// decisions buffer; rows of lanes that keep every token are left alone.
// ---------------------------------------------------------------------------------------------
struct Measure {
  uint32_t count;
  float mass;
};
constexpr uint32_t kEndThreads = 1024;
struct EndScratch {
  float mass[16][kEndThreads];
  uint32_t count[16][kEndThreads];
  float binMass[16];
  uint32_t binCount[16];
};
// One scan of the row: the 16-bin histogram of `digit(token, key)` (0..15, or 16 to leave a token
// out) over the selectable tokens at or before `end`, into scratch.binCount / binMass.
template <class Digit>
__device__ __forceinline__ void end_histogram(const float *x, uint32_t vocabulary, Mass mass, float inverse, OrderEnd end, Digit digit,
                                              EndScratch &scratch, uint32_t tid) {
#pragma unroll
  for (uint32_t b = 0; b < 16; ++b) {
    scratch.mass[b][tid] = 0.f;
    scratch.count[b][tid] = 0u;
  }
  for (uint32_t token = tid; token < vocabulary; token += kEndThreads) {
    const float value = x[token];
    if (unselectable(value)) continue;
    const uint32_t key = logit_key(value);
    if (!at_or_before(key, token, end)) continue;
    const uint32_t b = digit(token, key);
    if (b >= 16u) continue;
    scratch.mass[b][tid] += expf((value - mass.maximum) * inverse);
    scratch.count[b][tid] += 1u;
  }
  __syncthreads();
  // Wavefront w sums bin w: a lane its sixteen threads in order, the lanes in a fixed butterfly.
  const uint32_t lane = tid & 63u, b = tid >> 6;
  float m = 0.f;
  uint32_t c = 0;
#pragma unroll
  for (uint32_t i = 0; i < kEndThreads / 64u; ++i) {
    m += scratch.mass[b][lane + 64u * i];
    c += scratch.count[b][lane + 64u * i];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    m += __shfl_xor(m, o, 64);
    c += uint32_t(__shfl_xor(int(c), o, 64));
  }
  if (lane == 0) {
    scratch.binMass[b] = m;
    scratch.binCount[b] = c;
  }
  __syncthreads();
}
// The last token kept of the tokens at or before `end` (of which `all` measures everything), in
// order until their count exceeds `countTarget` (ByMass false) or their mass `massTarget` (ByMass
// true); `kept` becomes the measure of the kept tokens. Every thread returns the same.
template <bool ByMass>
__device__ OrderEnd select_last(const float *x, uint32_t vocabulary, Mass mass, float inverse, OrderEnd end, uint32_t countTarget,
                                float massTarget, Measure &kept, EndScratch &scratch, uint32_t tid) {
  auto exceeded = [&](Measure m) { return ByMass ? m.mass > massTarget : m.count > countTarget; };
  Measure above{0u, 0.f};
  uint32_t prefix = 0, tied = 0;
  for (int shift = 28; shift >= 0; shift -= 4) {
    const uint32_t high = shift == 28 ? 0u : prefix >> (shift + 4);
    end_histogram(x, vocabulary, mass, inverse, end,
                  [&](uint32_t, uint32_t key) { return shift != 28 && (key >> (shift + 4)) != high ? 16u : (key >> shift) & 15u; }, scratch, tid);
    int chosen = -1, lowest = -1;
    Measure cumulative = above;
    for (int b = 15; b >= 0 && chosen < 0; --b) {
      if (!scratch.binCount[b]) continue;
      const Measure next{cumulative.count + scratch.binCount[b], cumulative.mass + scratch.binMass[b]};
      lowest = b;
      if (exceeded(next)) chosen = b;
      else cumulative = next;
    }
    if (chosen < 0) {
      // The target is never exceeded: at the first pass every token stays; below it (a bin's mass and
      // its parts' may round apart) the search ends in the last bin that holds a token.
      if (shift == 28 || lowest < 0) {
        kept = cumulative;
        __syncthreads();
        return end;
      }
      chosen = lowest;
      cumulative = {cumulative.count - scratch.binCount[lowest], cumulative.mass - scratch.binMass[lowest]};
    }
    above = cumulative;
    prefix |= uint32_t(chosen) << shift;
    tied = scratch.binCount[chosen];
    __syncthreads();  // every thread has read the bins before the next pass clears them
  }
  // `tied` tokens share the key `prefix` and one weight: as many of them stay as the target takes.
  const float weight = expf((key_logit(prefix) - mass.maximum) * inverse);
  uint32_t keep;
  if (ByMass) {
    keep = weight > 0.f ? uint32_t(fminf(fmaxf((massTarget - above.mass) / weight, 0.f), float(tied))) : tied;
    keep = min(max(keep, 1u), tied);
    while (keep > 1u && above.mass + float(keep - 1u) * weight > massTarget) --keep;
    while (keep < tied && !(above.mass + float(keep) * weight > massTarget)) ++keep;
  } else {
    keep = min(max(countTarget + 1u - above.count, 1u), tied);
  }
  kept = {above.count + keep, above.mass + float(keep) * weight};
  OrderEnd last{prefix, 0xFFFFFFFFu};
  if (keep < tied) {
    // The keep-th smallest id of the tied tokens at or before `end`, by the same descent over ids.
    uint32_t bits = 4;
    while (bits < 32 && (vocabulary - 1u) >> bits) bits += 4;
    uint32_t id = 0, before = 0;
    for (int shift = int(bits) - 4; shift >= 0; shift -= 4) {
      const uint32_t high = shift + 4 >= 32 ? 0u : id >> (shift + 4);
      end_histogram(x, vocabulary, mass, inverse, end,
                    [&](uint32_t token, uint32_t key) {
                      return key != prefix || (shift + 4 < 32 && (token >> (shift + 4)) != high) ? 16u : (token >> shift) & 15u;
                    },
                    scratch, tid);
      uint32_t chosen = 15;
      for (uint32_t b = 0; b < 16; ++b) {
        if (before + scratch.binCount[b] >= keep) {
          chosen = b;
          break;
        }
        before += scratch.binCount[b];
      }
      id |= chosen << shift;
      __syncthreads();
    }
    last.last = id;
  }
  return last;
}

// A row whose end lies among its heaviest kEndCandidates tokens, which is nearly every row of a policy in use, is
// decided from them alone. The row is read twice: once to count its tokens in bins of (maximum - logit) / temperature, a
// sixteenth of an e-fold each, and once to gather those of the bins that are sure to hold the end. They are sorted by
// (logit, id) in LDS; the count and the running mass in that order are what top_k and top_p cut. Any other row (a
// nucleus of many thousand tokens) takes the descent above, a scan of the row a digit. What bounds the pass is one
// compute unit's reading of the row: 24 rows of 151936 logits under min_p 0.02, top_k 64 and top_p 0.95 took 1244 us by
// the descent of 256 threads, 39 us this way with every token keyed and 27 as it is.
constexpr uint32_t kEndCandidates = 8192, kEndBins = 512;
constexpr float kEndBinsPerFold = 16.f;
struct EndSelection {
  uint64_t order[kEndCandidates];  // (key, ~id), descending once sorted
  uint32_t bins[kEndBins];
  float waveMass[kEndThreads / 64u];
  float total;
  uint32_t selectable, gathered, cut, candidates, keep;
};
union EndShared {
  EndScratch descent;
  EndSelection selection;
};
// Calls all(four) of every four tokens of the row, a load whatever the row's alignment, and take(value, token) of the tokens
// of a four that holds a value at or above `floor` (past the row's end the values are -infinity). Few tokens pass a floor, so
// a scan costs what it does of every token: with the row's key, its comparison and a branch for each of them a row of 151936
// logits took 10 us a scan of its compute unit's vector ALUs, more than the 4 us of reading it.
template <class All, class Take>
__device__ __forceinline__ void end_scan(const float *x, uint32_t vocabulary, uint32_t tid, float floor, All all, Take take) {
  typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_unaligned;
  const f32x4_unaligned *v = reinterpret_cast<const f32x4_unaligned *>(x);
  const uint32_t vectors = vocabulary / 4u;
  auto four = [&](f32x4_unaligned held, uint32_t first) {
    all(held);
    if (!(fmaxf(fmaxf(held.x, held.y), fmaxf(held.z, held.w)) >= floor)) return;   // (a NaN is no maximum of others)
    take(held.x, first);
    take(held.y, first + 1u);
    take(held.z, first + 2u);
    take(held.w, first + 3u);
  };
  constexpr uint32_t kAhead = 8;
  for (uint32_t base = tid; base < vectors; base += kAhead * kEndThreads) {
    f32x4_unaligned held[kAhead];
#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i) {
      const uint32_t at = base + i * kEndThreads;
      held[i] = at < vectors ? v[at] : f32x4_unaligned{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    }
#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i) four(held[i], 4u * (base + i * kEndThreads));
  }
  if (tid < vocabulary % 4u) four(f32x4_unaligned{x[4u * vectors + tid], -INFINITY, -INFINITY, -INFINITY}, 4u * vectors + tid);
}
__device__ __forceinline__ uint32_t end_bin(float value, float maximum, float inverse) {
  return uint32_t(min(int((maximum - value) * inverse * kEndBinsPerFold), int(kEndBins) - 1));  // rises as the logit falls
}

__global__ __launch_bounds__(kEndThreads) void decode_sample_distribution_end(const float *__restrict__ logits,
                                                                              const float *__restrict__ masses,
                                                                              uint32_t *__restrict__ decisions, TargetSamplingParams p) {
  __shared__ EndShared shared;
  EndSelection &s = shared.selection;
  const uint32_t row = blockIdx.x, tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, laneIndex = lane_of_row(p, row);
  if (!((p.truncating_mask >> laneIndex) & 1u)) return;
  const float temperature = p.temperature[laneIndex], inverse = 1.0f / temperature;
  const float *x = logits + size_t(row) * p.logits_stride;
  const float minP = p.min_p[laneIndex], topP = p.top_p[laneIndex];
  const uint32_t topK = p.top_k[laneIndex];
  const float maximum = wave_max(masses[2u * (row * SAMPLING_SHARDS + lane % SAMPLING_SHARDS)]);
  // what min_p keeps: the tokens at or above the logit that weighs min_p of the heaviest
  const float floor = minP > 0.f ? fminf(maximum + temperature * logf(minP), maximum) : -INFINITY;
  const uint32_t lowest = logit_key(floor);
  for (uint32_t b = tid; b < kEndBins; b += kEndThreads) s.bins[b] = 0;
  if (wave == 0) {
    const float total = row_mass(masses, row, inverse).sum;
    if (lane == 0) {
      s.total = total;
      s.selectable = s.gathered = s.candidates = 0;
      s.cut = kEndBins - 1u;
    }
  }
  __syncthreads();
  uint32_t selectable = 0;
  end_scan(x, p.vocabulary, tid, floor,
           [&](auto held) {
#pragma unroll
             for (int e = 0; e < 4; ++e) selectable += unselectable(held[e]) ? 0u : 1u;
           },
           [&](float value, uint32_t) {
             if (unselectable(value)) return;
             if (logit_key(value) >= lowest) atomicAdd(&s.bins[end_bin(value, maximum, inverse)], 1u);
           });
  selectable = wave_sum(selectable);
  if (lane == 0) atomicAdd(&s.selectable, selectable);
  __syncthreads();
  // The first bin that ends past top_k tokens, or past a mass that exceeds top_p of the row's, a token of bin b weighing
  // at least exp(-(b + 1) / 16); a nucleus of what min_p leaves needs the mass of all of it.
  if (wave == 0) {
    uint32_t count[kEndBins / 64u], sum = 0;
    float mass[kEndBins / 64u], massSum = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < kEndBins / 64u; ++i) {
      const uint32_t b = lane * (kEndBins / 64u) + i, c = s.bins[b];
      sum += c;
      massSum += b + 1u < kEndBins ? float(c) * expf(-float(b + 1u) / kEndBinsPerFold) * 0.999f : 0.f;
      count[i] = sum;
      mass[i] = massSum;
    }
    uint32_t before = sum;
    float massBefore = massSum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t c = uint32_t(__shfl_up(int(before), o, 64));
      const float m = __shfl_up(massBefore, o, 64);
      if (int(lane) >= o) {
        before += c;
        massBefore += m;
      }
    }
    const uint32_t all = uint32_t(__shfl(int(before), 63, 64));
    before -= sum;
    massBefore -= massSum;
    const bool byCount = topK && topK < all, byMass = !byCount && minP <= 0.f && topP < 1.0f;
    uint32_t cut = kEndBins - 1u;
#pragma unroll
    for (int i = int(kEndBins / 64u) - 1; i >= 0; --i) {
      const bool past = byCount ? before + count[i] >= topK : byMass && massBefore + mass[i] > 1.001f * topP * s.total;
      if (past) cut = lane * (kEndBins / 64u) + uint32_t(i);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cut = min(cut, uint32_t(__shfl_xor(int(cut), o, 64)));
    if (lane == cut / (kEndBins / 64u)) {
      uint32_t upTo = 0;
#pragma unroll
      for (uint32_t i = 0; i < kEndBins / 64u; ++i) upTo = i == cut % (kEndBins / 64u) ? before + count[i] : upTo;
      s.cut = cut;
      s.candidates = upTo;
    }
    if (lane == 0) s.keep = all;
  }
  __syncthreads();
  const uint32_t all = s.keep, admitted = s.selectable, candidates = s.candidates, cut = s.cut;
  const float rowTotal = s.total;
  const bool minCuts = minP > 0.f && all < admitted;
  OrderEnd end{0u, 0u};
  Measure kept{all, 0.f};
  if (candidates <= kEndCandidates) {
    const uint32_t slots = candidates <= 1u ? 1u : 1u << (32u - uint32_t(__builtin_clz(candidates - 1u)));
    for (uint32_t i = candidates + tid; i < slots; i += kEndThreads) s.order[i] = 0;
    // A token of bin `cut` or before lies at or above this: the bin's far edge, and further out by more than the roundings of
    // end_bin and of this line move it. (An infinite maximum makes it NaN, which fmaxf drops.)
    const float edge = cut + 1u < kEndBins ? maximum - float(cut + 1u) / kEndBinsPerFold * temperature * 1.0001f - fabsf(maximum) * 1e-6f : -INFINITY;
    end_scan(x, p.vocabulary, tid, fmaxf(floor, edge), [](auto) {},
             [&](float value, uint32_t token) {
               if (unselectable(value)) return;
               const uint32_t key = logit_key(value);
               if (key < lowest || end_bin(value, maximum, inverse) > cut) return;
               s.order[atomicAdd(&s.gathered, 1u)] = uint64_t(key) << 32 | uint64_t(~token);
             });
    __syncthreads();
    // bitonic, descending (the order they were gathered in leaves no trace: no two are equal)
    for (uint32_t size = 2; size <= slots; size <<= 1)
      for (uint32_t stride = size / 2; stride; stride >>= 1) {
        for (uint32_t i = tid; i < slots / 2; i += kEndThreads) {
          const uint32_t low = 2u * i - (i & (stride - 1u)), high = low + stride;
          const uint64_t a = s.order[low], b = s.order[high];
          if ((a < b) == ((low & size) == 0u)) {
            s.order[low] = b;
            s.order[high] = a;
          }
        }
        __syncthreads();
      }
    const bool countCuts = topK && topK < all;
    kept.count = countCuts ? topK : all;
    // The running mass, a thread eight tokens in order; of the kept tokens past the candidates (a nucleus of the whole
    // row) the row's total says what they weigh.
    constexpr uint32_t kEach = kEndCandidates / kEndThreads;
    const uint32_t listed = min(kept.count, candidates);
    float mine[kEach], sum = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < kEach; ++i) {
      const uint32_t at = tid * kEach + i;
      sum += at < listed ? expf((key_logit(uint32_t(s.order[at] >> 32)) - maximum) * inverse) : 0.f;
      mine[i] = sum;
    }
    float before = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float m = __shfl_up(before, o, 64);
      if (int(lane) >= o) before += m;
    }
    if (lane == 63u) s.waveMass[wave] = before;
    if (tid == 0) s.keep = 0xFFFFFFFFu;
    __syncthreads();
    before -= sum;
    float base = 0.f, total = 0.f;
    for (uint32_t w = 0; w < kEndThreads / 64u; ++w) {
      if (w == wave) base = total;
      total += s.waveMass[w];
    }
    kept.mass = candidates < kept.count ? rowTotal : total;
    const float nucleus = topP * kept.mass;
    if (topP < 1.0f) {
#pragma unroll
      for (int i = int(kEach) - 1; i >= 0; --i) {
        const uint32_t at = tid * kEach + uint32_t(i);
        // (a running mass that rounding turned back does not end the nucleus twice: the first token past it does)
        if (at < listed && base + (before + mine[i]) > nucleus) atomicMin(&s.keep, at + 1u);
      }
    }
    __syncthreads();
    const uint32_t nucleusEnd = s.keep;
    const bool massCuts = nucleusEnd != 0xFFFFFFFFu;
    if (massCuts) kept.count = nucleusEnd;
    if (minCuts) end = {lowest, 0xFFFFFFFFu};
    if (countCuts || massCuts) {
      const uint64_t last = s.order[kept.count - 1u];
      const uint32_t key = uint32_t(last >> 32);
      // every token of the last one's key is among the candidates
      const bool tied = kept.count < candidates && uint32_t(s.order[kept.count] >> 32) == key;
      end = {key, tied ? ~uint32_t(last) : 0xFFFFFFFFu};
    }
    if (massCuts && tid == (nucleusEnd - 1u) / kEach) {
      float at = 0.f;
#pragma unroll
      for (uint32_t i = 0; i < kEach; ++i) at = i == (nucleusEnd - 1u) % kEach ? mine[i] : at;
      s.total = base + (before + at);
    }
    __syncthreads();
    if (massCuts) kept.mass = s.total;
  } else {
    EndScratch &scratch = shared.descent;
    __syncthreads();
    const Mass mass{maximum, rowTotal};
    end_histogram(x, p.vocabulary, mass, inverse, end, [&](uint32_t, uint32_t key) { return key >= lowest ? 1u : 0u; }, scratch, tid);
    kept = {scratch.binCount[1], scratch.binMass[1]};
    __syncthreads();
    if (minCuts) end = {lowest, 0xFFFFFFFFu};
    if (topK && topK < kept.count) end = select_last<false>(x, p.vocabulary, mass, inverse, end, topK - 1u, 0.f, kept, scratch, tid);
    if (topP < 1.0f) end = select_last<true>(x, p.vocabulary, mass, inverse, end, 0u, topP * kept.mass, kept, scratch, tid);
  }
  if (tid == 0) {
    uint32_t *words = decisions + size_t(row) * SAMPLING_DECISION_WORDS;
    words[SAMPLING_END_KEY] = end.key;
    words[SAMPLING_END_LAST] = end.last;
    words[SAMPLING_END_MASS] = __builtin_bit_cast(uint32_t, kept.mass);
    words[SAMPLING_END_COUNT] = kept.count;
  }
}
SP_REGISTER_KERNEL("decode_sample_distribution_end", &decode_sample_distribution_end);

constexpr uint32_t kChunks = SAMPLING_THREADS;  // chunks of a range, one per thread
__device__ __forceinline__ uint32_t range_tokens(uint32_t vocabulary) {
  return (vocabulary + SAMPLING_RANGES - 1) / SAMPLING_RANGES;
}
__device__ __forceinline__ uint32_t chunk_tokens(uint32_t vocabulary) { return (range_tokens(vocabulary) + kChunks - 1) / kChunks; }

// Grid (rows * SAMPLING_RANGES / 4), 256 threads: each wavefront sums one range; thread 0 of the
// row's first workgroup also records the rejection test. ranges [row][SAMPLING_RANGES];
// decisions [row][2]: the accepted child token or SAMPLING_NO_TOKEN when the row must draw, and
// whether it draws from the residual (1) or from p (0). uniforms [row][2]: the row's draw, its child's test.
__global__ __launch_bounds__(256) void decode_sample_residual_ranges(const float *__restrict__ logits, const float *__restrict__ draft,
                                                                     const float *__restrict__ masses, const float *__restrict__ uniforms,
                                                                     const AttentionTreeRow *__restrict__ tree,
                                                                     const uint32_t *__restrict__ input_tokens,
                                                                     float *__restrict__ ranges, uint32_t *__restrict__ decisions,
                                                                     TargetSamplingParams p) {
  constexpr uint32_t kPerRow = SAMPLING_RANGES / 4, kStagedRange = 1024;
  __shared__ float staged[4][kStagedRange];
  const uint32_t row = blockIdx.x / kPerRow, range = (blockIdx.x % kPerRow) * 4u + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
  const uint32_t laneIndex = lane_of_row(p, row);
  const float inverse = 1.0f / p.temperature[laneIndex];
  const Kept kept = row_kept(masses, decisions, row, inverse, (p.truncating_mask >> laneIndex) & 1u);
  const float *x = logits + size_t(row) * p.logits_stride, *q = draft + size_t(row) * p.logits_stride;
  // a row that tests candidate children sums the ranges of its whole distribution: the draw kernel does the tests
  const uint32_t child = p.candidate_children ? SAMPLING_NO_TOKEN : child_token(p, tree, input_tokens, row);
  bool rejected = false;
  if (child != SAMPLING_NO_TOKEN && child < p.vocabulary) {
    // accept iff u_child * q < p (sampling.metal:790-800)
    const float pc = kept_weight(x[child], child, kept, inverse) / kept.mass.sum;
    rejected = !(uniforms[2 * row + 1] * q[child] < pc);
    if (blockIdx.x % kPerRow == 0 && threadIdx.x == 0) {
      decisions[SAMPLING_DECISION_WORDS * row] = rejected ? SAMPLING_NO_TOKEN : child;
      decisions[SAMPLING_DECISION_WORDS * row + 1] = rejected ? 1u : 0u;
    }
  } else if (blockIdx.x % kPerRow == 0 && threadIdx.x == 0) {
    decisions[SAMPLING_DECISION_WORDS * row] = SAMPLING_NO_TOKEN;
    decisions[SAMPLING_DECISION_WORDS * row + 1] = 0u;
  }
  if (child != SAMPLING_NO_TOKEN && child < p.vocabulary && !rejected) return;  // accepted: nothing to draw
  // The range's residual: a lane sums its tokens in id order, the lanes are added in order. The tokens are weighed 64
  // neighbours at a time and handed to their lanes through LDS (24 rows of 151936: 19.1 us with each lane's tokens read where
  // it sums them, 40 bytes from the next lane's, 14.5 so; the same sums); a range that LDS does not hold, of a vocabulary past
  // 262144, is still read that way.
  const uint32_t size = range_tokens(p.vocabulary), begin = range * size, end = min(p.vocabulary, begin + size);
  const uint32_t per = (size + 63u) / 64u;
  float sum = 0.f;
  if (size <= kStagedRange) {
    float *mine = staged[threadIdx.x >> 6];
    constexpr uint32_t kAhead = 5;
    for (uint32_t first = lane; first < size; first += 64u * kAhead) {
      float logit[kAhead], drafted[kAhead];
#pragma unroll
      for (uint32_t i = 0; i < kAhead; ++i) {
        const uint32_t at = min(begin + first + 64u * i, p.vocabulary - 1u);
        logit[i] = x[at];
        drafted[i] = rejected ? q[at] : 0.f;
      }
#pragma unroll
      for (uint32_t i = 0; i < kAhead; ++i) {
        const uint32_t at = first + 64u * i, token = begin + at;
        if (at < size) mine[at] = token < end ? residual_of(logit[i], token, drafted[i], kept, inverse, rejected) : 0.f;
      }
    }
    wave_lds_fence();
    for (uint32_t i = lane * per; i < min(lane * per + per, size); ++i) sum += mine[i];
  } else {
    sum = lane_residual(x, q, begin + lane * per, per, end, kept, inverse, rejected);
  }
  float total = 0.f;
#pragma unroll
  for (int l = 0; l < 64; ++l) total += lane_value_of(sum, l);
  if (lane == 0) ranges[row * SAMPLING_RANGES + range] = total;
}
SP_REGISTER_KERNEL("decode_sample_residual_ranges", &decode_sample_residual_ranges);

// The wavefront's 64 values, in every lane, for a walk in lane order: once through LDS, where a shuffle a step would wait for
// each. `staged` is the wavefront's own.
__device__ __forceinline__ void wave_values(float mine, float *staged, float (&values)[64]) {
  wave_lds_fence();   // (what the walk before read)
  staged[threadIdx.x & 63u] = mine;
  wave_lds_fence();
#pragma unroll
  for (uint32_t i = 0; i < 16; ++i) {
    const float4 v = reinterpret_cast<const float4 *>(staged)[i];
    values[4 * i] = v.x;
    values[4 * i + 1] = v.y;
    values[4 * i + 2] = v.z;
    values[4 * i + 3] = v.w;
  }
}

// The running sums of `count` values of LDS, a multiple of four, in their order and from `start`: before[i] what lies before
// value i, before[count] all of it. One lane's chain of additions and nothing else: what a walk in order asks of each step
// (is the point passed, is this the last with weight) the lanes then ask of all of them at once. (24 rows' draws: 27 us with
// walks that asked at each step, unrolled into 20 KB of instructions; 10.6 so. The same sums and the same token.)
__device__ __forceinline__ void running_sums(const float *values, float *before, uint32_t count, float start) {
  wave_lds_fence();   // (the values are written, and what was read of `before`)
  if ((threadIdx.x & 63u) == 0) {
    float sum = start;
#pragma unroll 4
    for (uint32_t i = 0; i < count / 4u; ++i) {
      const float4 v = reinterpret_cast<const float4 *>(values)[i];
      float4 b;
      b.x = sum;
      b.y = b.x + v.x;
      b.z = b.y + v.y;
      b.w = b.z + v.z;
      sum = b.w + v.w;
      reinterpret_cast<float4 *>(before)[i] = b;
    }
    before[count] = sum;
  }
  wave_lds_fence();
}
// Of values whose running sums are `before`: the first that the point lies inside, or the last that has weight (0 if none has).
template <uint32_t Count> __device__ __forceinline__ uint32_t value_at(const float *values, const float *before, float point) {
  uint32_t hit = Count, lastWeighted = 0;
#pragma unroll
  for (uint32_t i = 0; i < Count; i += 64u) {
    const uint32_t j = i + (threadIdx.x & 63u);
    const uint64_t passed = __ballot(point < before[j] + values[j]), weighted = __ballot(values[j] > 0.f);
    if (hit == Count && passed) hit = i + uint32_t(__builtin_ctzll(passed));
    if (weighted) lastWeighted = i + 63u - uint32_t(__builtin_clzll(weighted));
  }
  return hit == Count ? lastWeighted : hit;
}

// Grid (rows), 64 threads: the row's selection. A sampled row whose child was accepted selects it;
// otherwise it draws at point = u_row * sum of the ranges, from the residual when its child was
// rejected (decisions[2 row + 1] == 1) and from p itself when it has no child.
__global__ __launch_bounds__(64) void decode_sample_draw(const float *__restrict__ logits, const float *__restrict__ draft,
                                                         const float *__restrict__ masses, const float *__restrict__ uniforms,
                                                         const float *__restrict__ ranges, const uint32_t *__restrict__ decisions,
                                                         uint32_t *__restrict__ tokens, TargetSamplingParams p) {
  const uint32_t row = blockIdx.x, lane = threadIdx.x;
  const uint32_t laneIndex = lane_of_row(p, row);
  if (!((p.sampling_mask >> laneIndex) & 1u)) return;  // a greedy lane keeps its argmax
  const uint32_t decision = decisions[SAMPLING_DECISION_WORDS * row];
  if (decision != SAMPLING_NO_TOKEN) {
    if (lane == 0) tokens[row] = decision;
    return;
  }
  const bool rejected = decisions[SAMPLING_DECISION_WORDS * row + 1] == 1u;
  const float inverse = 1.0f / p.temperature[laneIndex];
  const Kept kept = row_kept(masses, decisions, row, inverse, (p.truncating_mask >> laneIndex) & 1u);
  const float *x = logits + size_t(row) * p.logits_stride, *q = draft + size_t(row) * p.logits_stride;
  const float *r = ranges + row * SAMPLING_RANGES;
  // the ranges in LDS: the sums walk them in order without a trip to memory each
  __shared__ __align__(16) float weights[SAMPLING_RANGES], before[SAMPLING_RANGES + 4];
#pragma unroll
  for (uint32_t i = 0; i < SAMPLING_RANGES / 64u; ++i) weights[lane + 64u * i] = r[lane + 64u * i];
  running_sums(weights, before, SAMPLING_RANGES, 0.f);
  const float total = before[SAMPLING_RANGES];
  if (!(total > 0.f)) {
    if (lane == 0) tokens[row] = SAMPLING_NO_TOKEN;
    return;
  }
  // The range that holds the point; the last weighted range on a rounding shortfall.
  const float point = uniforms[2 * row] * total;
  const uint32_t hit = value_at<SAMPLING_RANGES>(weights, before, point);
  float target = point - before[hit];
  // Its lanes' chunks, as the ranges kernel summed them, walked in lane order.
  const uint32_t size = range_tokens(p.vocabulary), begin = hit * size, end = min(p.vocabulary, begin + size);
  const uint32_t per = (size + 63u) / 64u;
  const float sum = lane_residual(x, q, begin + lane * per, per, end, kept, inverse, rejected);
  wave_lds_fence();
  weights[lane] = sum;
  running_sums(weights, before, 64u, 0.f);
  const uint32_t chunk = value_at<64u>(weights, before, target);
  target -= before[chunk];
  // The chunk's tokens, weighed a lane each and walked in id order.
  uint32_t selected = SAMPLING_NO_TOKEN, lastToken = SAMPLING_NO_TOKEN;
  float walked = 0.f;
  for (uint32_t i0 = 0; i0 < per && selected == SAMPLING_NO_TOKEN; i0 += 64u) {
    const uint32_t first = begin + chunk * per + i0, own = first + lane;
    const bool live = i0 + lane < per && own < end;
    const float weight = live ? residual_of(x[own], own, rejected ? q[own] : 0.f, kept, inverse, rejected) : 0.f;
    wave_lds_fence();
    weights[lane] = weight;
    running_sums(weights, before, 64u, walked);
    const uint64_t weighted = __ballot(weight > 0.f), passed = __ballot(weight > 0.f && target < before[lane] + weight);
    if (passed) selected = first + uint32_t(__builtin_ctzll(passed));
    if (weighted) lastToken = first + 63u - uint32_t(__builtin_clzll(weighted));
    walked = before[64];
  }
  if (lane == 0) tokens[row] = selected != SAMPLING_NO_TOKEN ? selected : lastToken;
}
SP_REGISTER_KERNEL("decode_sample_draw", &decode_sample_draw);

// decode_sample_draw_children (the rule of the reference's vocabulary_draw with children, sampling.metal:697-880): grid
// (rows), 64 threads. A sampled row of a tree block tests the children its draft drew among its SAMPLING_CANDIDATES
// candidates -- ids [row][16], their draft probabilities q [row][16], the candidate indices drawn in order draws
// [row][4] (bytes, SAMPLING_NO_DRAW past them), a uniform a child child_uniforms [row][4] -- by recursive rejection
// sampling without replacement: child c is selected iff u_c q_c < p_c; a rejection leaves the target its residual
// max(p - q, 0) over the candidates and its mass outside them, renormalized, and the draft its rest, renormalized. A
// row that selects none draws at u_row of the last residual: a candidate in index order, or past them a token
// outside them in id order by the target's own weights. The ranges hold the row's kept weights (the ranges kernel
// ran without a child); the candidates' weights leave them here. Lanes 0..15 weigh a candidate each, lane 0 decides,
// the wavefront walks the drawn range.
__global__ __launch_bounds__(64) void decode_sample_draw_children(const float *__restrict__ logits, const float *__restrict__ masses,
                                                                  const float *__restrict__ uniforms, const float *__restrict__ ranges,
                                                                  const uint32_t *__restrict__ decisions,
                                                                  const uint32_t *__restrict__ candidate_ids,
                                                                  const float *__restrict__ candidate_q,
                                                                  const uint8_t *__restrict__ draws,
                                                                  const float *__restrict__ child_uniforms,
                                                                  uint32_t *__restrict__ tokens, TargetSamplingParams p) {
  constexpr uint32_t K = SAMPLING_CANDIDATES;
  __shared__ float rangeWeight[SAMPLING_RANGES];
  __shared__ float candidateWeight[K];
  __shared__ __align__(16) float staged[64];
  __shared__ uint32_t excludedIds[K];
  __shared__ uint32_t decided[4];  // selected (1) or walking (0), token or range, target bits, excluding
  const uint32_t row = blockIdx.x, lane = threadIdx.x;
  const uint32_t laneIndex = lane_of_row(p, row);
  if (!((p.sampling_mask >> laneIndex) & 1u)) return;  // a greedy lane keeps its argmax
  const float inverse = 1.0f / p.temperature[laneIndex];
  const Kept kept = row_kept(masses, decisions, row, inverse, (p.truncating_mask >> laneIndex) & 1u);
  const float *x = logits + size_t(row) * p.logits_stride;
  const uint32_t size = range_tokens(p.vocabulary);
  for (uint32_t j = lane; j < SAMPLING_RANGES; j += 64u) rangeWeight[j] = ranges[row * SAMPLING_RANGES + j];
  if (lane < K) {
    const uint32_t id = candidate_ids[row * K + lane];
    excludedIds[lane] = id;
    candidateWeight[lane] = id < p.vocabulary ? kept_weight(x[id], id, kept, inverse) : 0.f;
  }
  __syncthreads();
  if (lane == 0) {
    float total = 0.f;
    for (uint32_t j = 0; j < SAMPLING_RANGES; ++j) total += rangeWeight[j];
    bool selected = false, excluding = false;
    uint32_t token = SAMPLING_NO_TOKEN;
    float target = uniforms[2 * row] * total;
    const uint8_t *drawn = draws + row * SAMPLING_TREE_CHILDREN;
    if (!(total > 0.f)) {
      selected = true;  // nothing selectable: the sentinel
    } else if (drawn[0] != SAMPLING_NO_DRAW) {
      float pc[K], qc[K];
      for (uint32_t i = 0; i < K; ++i) {
        const uint32_t id = excludedIds[i];
        const float weight = candidateWeight[i];
        if (id < p.vocabulary) rangeWeight[id / size] = fmaxf(rangeWeight[id / size] - weight, 0.f);
        pc[i] = weight / total;
        qc[i] = candidate_q[row * K + i];
      }
      float outsideWeight = 0.f;
      for (uint32_t j = 0; j < SAMPLING_RANGES; ++j) outsideWeight += rangeWeight[j];
      float outside = outsideWeight / total;
      for (uint32_t child = 0; child < SAMPLING_TREE_CHILDREN && !selected; ++child) {
        const uint32_t c = drawn[child];
        if (c >= K) break;
        // a dynamic index into a register array would spill: pick the child's p and q by comparison
        float pChild = 0.f, qChild = 0.f;
        for (uint32_t i = 0; i < K; ++i) { pChild = i == c ? pc[i] : pChild; qChild = i == c ? qc[i] : qChild; }
        if (child_uniforms[row * SAMPLING_TREE_CHILDREN + child] * qChild < pChild) {
          selected = true;
          token = excludedIds[c];
          break;
        }
        float residual = outside;
        for (uint32_t i = 0; i < K; ++i) residual += fmaxf(pc[i] - qc[i], 0.f);
        if (!(residual > 0.f)) break;
        for (uint32_t i = 0; i < K; ++i) pc[i] = fmaxf(pc[i] - qc[i], 0.f) / residual;
        outside /= residual;
        float rest = 0.f;
        for (uint32_t i = 0; i < K; ++i) { qc[i] = i == c ? 0.f : qc[i]; rest += qc[i]; }
        for (uint32_t i = 0; rest > 0.f && i < K; ++i) qc[i] /= rest;
      }
      if (!selected) {
        float inside = 0.f;
        for (uint32_t i = 0; i < K; ++i) inside += pc[i];
        const float point = uniforms[2 * row] * (inside + outside);
        float cumulative = 0.f;
        uint32_t last = K;
        for (uint32_t i = 0; i < K && !(point < cumulative); ++i)
          if (pc[i] > 0.f) {
            last = i;
            cumulative += pc[i];
          }
        if (last < K && (point < cumulative || !(outside > 0.f))) {
          selected = true;
          token = excludedIds[last];
        } else {
          excluding = true;
          target = (point - inside) / outside * outsideWeight;
        }
      }
    }
    uint32_t hit = 0;
    float within = 0.f;
    if (!selected) {
      // the first weighted range whose end lies past the target; the last weighted one on a rounding shortfall
      float cumulative = 0.f;
      for (uint32_t j = 0; j < SAMPLING_RANGES; ++j) {
        const float weight = rangeWeight[j];
        if (!(weight > 0.f)) continue;
        hit = j;
        within = target - cumulative;
        cumulative += weight;
        if (cumulative > target) break;
      }
    }
    decided[0] = selected ? 1u : 0u;
    decided[1] = selected ? token : hit;
    decided[2] = __builtin_bit_cast(uint32_t, within);
    decided[3] = excluding ? 1u : 0u;
  }
  __syncthreads();
  if (decided[0]) {
    if (lane == 0) tokens[row] = decided[1];
    return;
  }
  const uint32_t hit = decided[1];
  const bool excluding = decided[3] != 0u;
  float target = __builtin_bit_cast(float, decided[2]);
  auto weigh = [&](uint32_t token) {
    bool out = false;
    if (excluding)
      for (uint32_t i = 0; i < K; ++i) out = out || excludedIds[i] == token;
    return out ? 0.f : kept_weight(x[token], token, kept, inverse);
  };
  // the range's lanes' chunks, as the ranges kernel summed them (less the candidates), walked in lane order
  const uint32_t begin = hit * size, end = min(p.vocabulary, begin + size), per = (size + 63u) / 64u;
  float sum = 0.f;
  for (uint32_t i = 0; i < per; ++i) {
    const uint32_t token = begin + lane * per + i;
    if (token < end) sum += weigh(token);
  }
  uint32_t chunk = 64, lastChunk = 0;
  float chunkBefore = 0.f, lastChunkBefore = 0.f, cumulative = 0.f;
  float sums[64];
  wave_values(sum, staged, sums);
#pragma unroll
  for (int l = 0; l < 64; ++l) {
    const float c = sums[l];
    if (c > 0.f) { lastChunk = uint32_t(l); lastChunkBefore = cumulative; }
    if (chunk == 64 && c > 0.f && target < cumulative + c) { chunk = uint32_t(l); chunkBefore = cumulative; }
    cumulative += c;
  }
  if (chunk == 64) { chunk = lastChunk; chunkBefore = lastChunkBefore; }
  target -= chunkBefore;
  if (lane == 0) {
    uint32_t selected = SAMPLING_NO_TOKEN, lastToken = SAMPLING_NO_TOKEN;
    float walked = 0.f;
    for (uint32_t i = 0; i < per; ++i) {
      const uint32_t token = begin + chunk * per + i;
      if (token >= end) break;
      const float w = weigh(token);
      if (w > 0.f) lastToken = token;
      walked += w;
      if (selected == SAMPLING_NO_TOKEN && w > 0.f && target < walked) selected = token;
    }
    tokens[row] = selected != SAMPLING_NO_TOKEN ? selected : lastToken;
  }
}
SP_REGISTER_KERNEL("decode_sample_draw_children", &decode_sample_draw_children);

} // namespace splash::kernels

// ---- Greedy selection of packed logits rows without any allocation ------------------------------
// spo_sampling_greedy_rows_static (include/splash_ops.h) is the argmax pair above for callers that
// cannot allocate: the shards' partials live in a file-scope device array instead of a workspace.
// Host code never uses the array's name as an address: each device's copy is looked up once with
// hipGetSymbolAddress and that pointer is what the kernels get.
#include "backend/Internal.hpp"
#include "splash_ops.h"

#include <hip/hip_runtime.h>
#include <mutex>

namespace splash::kernels {
namespace {

struct GreedyPartial {
  float value;
  uint32_t index;
};
constexpr uint32_t kStaticRows = SPO_SAMPLING_STATIC_MAXIMUM_ROWS;
constexpr int kMaximumDevices = 64;
static __device__ __align__(256) unsigned char scratch[kStaticRows * SAMPLING_SHARDS * sizeof(GreedyPartial)];

std::mutex scratchMutex;
void *scratchOfDevice[kMaximumDevices];  // each device holds its own copy of the array, at its own address

// The current device's copy of the scratch array (looked up on the device's first call).
hipError_t deviceScratch(void **out) {
  int device = -1;
  hipError_t status = hipGetDevice(&device);
  if (status != hipSuccess) return status;
  if (device < 0 || device >= kMaximumDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(scratchMutex);
  if (!scratchOfDevice[device]) {
    void *address = nullptr;
    status = hipGetSymbolAddress(&address, HIP_SYMBOL(scratch));
    if (status != hipSuccess) return status;
    scratchOfDevice[device] = address;
  }
  *out = scratchOfDevice[device];
  return hipSuccess;
}

} // namespace
} // namespace splash::kernels

extern "C" sp_status spo_sampling_greedy_rows_static(const float *logits, uint32_t rows, uint32_t vocabulary, uint32_t logits_stride,
                                                     uint32_t *tokens, void *stream) {
  using namespace splash::kernels;
  auto fail = [](sp_status code, const std::string &message) {
    splash::hipbackend::setLastError(message);
    return code;
  };
  if (!logits || !tokens) return fail(SP_INVALID_ARGUMENT, "null logits or tokens");
  if (!rows || rows > kStaticRows)
    return fail(SP_INVALID_ARGUMENT, "the static greedy selection takes 1 to " + std::to_string(kStaticRows) + " rows");
  if (!vocabulary || logits_stride < vocabulary) return fail(SP_INVALID_ARGUMENT, "a logits row holds its vocabulary");
  void *memory = nullptr;
  hipError_t status = deviceScratch(&memory);
  if (status != hipSuccess) return fail(SP_BACKEND_ERROR, std::string("hipGetSymbolAddress: ") + hipGetErrorString(status));
  // Every (row, shard) partial of this call is written by the first kernel before the second reads
  // it, so nothing of an earlier call's contents is read and nothing needs clearing.
  float *values = static_cast<float *>(memory);
  uint32_t *indices = reinterpret_cast<uint32_t *>(values + size_t(kStaticRows) * SAMPLING_SHARDS);
  TargetSamplingParams p{};
  p.vocabulary = vocabulary;
  p.rows = rows;
  p.lanes = 1;
  p.logits_stride = logits_stride;
  p.lane[0] = SamplingLaneRows{0, rows};
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(decode_sample_argmax_sharded, dim3(rows * SAMPLING_SHARDS), dim3(256), 0, s, logits, values, indices, p);
  hipLaunchKernelGGL(decode_sample_argmax_reduce, dim3(rows), dim3(64), 0, s, values, indices, tokens, p);
  status = hipGetLastError();
  if (status != hipSuccess) return fail(SP_BACKEND_ERROR, std::string("launch: ") + hipGetErrorString(status));
  return SP_OK;
}
