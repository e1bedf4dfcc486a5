// The draft selector's tree growth (the reference's draft_select_tree, kernels/decode/sampling.metal:1357-1766; its rule,
// runtime/metal/abi/Sampling.h:209-241): over the candidates and edge scores draft_select_edges left, each lane grows a
// tree of up to 16 rows best first by the estimate that the target accepts the path to a row.
//
// One workgroup a lane. What does not depend on the tree (the distributions after every candidate, the lane's tempered ones
// and the estimates) is computed first, for all 97 of them side by side; then one wavefront grows the tree, a serial chain
// of up to 15 steps that is nothing but latency, so it holds the rows and the tree's open steps ("entries": from a row to a
// token one deeper, at most five a row) in its lanes' registers and reads them by lane number: no heap, no barrier, and no
// LDS write to wait for. The best entry is one 64-bit maximum over (estimate bits, complement of the entry's number),
// exactly "the largest estimate, the earlier entry among equal ones"; a draw is a 16-lane maximum over the Gumbel keys (a
// hash of the row's key and the candidate's token a lane). Sums whose order decides a float's bits (a distribution's mass)
// are taken in candidate order, as a sequential statement takes them, so the values agree with it to the rounding of exp
// and log alone. Eight lanes' trees of 16 rows: 61 -> 36 us (all of it in one wavefront, with LDS between the steps, before),
// -> 31.6 with four teams of threads on the distributions (6 us of the pass by now; a step of the growth is 1.6).
#include "abi/PagedAttention.h"
#include "abi/Sampling.h"
#include "backend/KernelRegistry.hpp"
#include "kernels/device_common.hpp"

namespace splash::kernels {
namespace {

constexpr uint32_t kPositions = DRAFT_PROPOSAL_TOKENS, kCandidates = DRAFT_CANDIDATES, kChildren = SAMPLING_TREE_CHILDREN;
constexpr uint32_t kRows = DRAFT_TREE_ROWS, kEntries = 96, kDead = 0xFFFFFFFFu, kChainEntry = 1u << 31;

__device__ __forceinline__ uint64_t mix64(uint64_t v) {  // the splitmix64 finalizer
  v = (v ^ (v >> 30)) * 0xbf58476d1ce4e5b9ull;
  v = (v ^ (v >> 27)) * 0x94d049bb133111ebull;
  return v ^ (v >> 31);
}
// The standard Gumbel of candidate `token` under a row of key `key`: of a uniform from the top 23 bits k of a hash of the
// two, (k + 0.5) / 2^23, which fp32 holds exactly, inside (0, 1).
__device__ __forceinline__ float gumbel_of(uint64_t key, uint32_t token) {
  const uint64_t v = mix64(key ^ 0xd1b54a32d192ed03ull * (uint64_t(token) + 1u));
  const float uniform = (float(uint32_t(v >> 41)) + 0.5f) * 0x1p-23f;
  return -logf(-logf(uniform));
}
__device__ __forceinline__ uint32_t order_bits(float value) {
  const uint32_t bits = __float_as_uint(value);
  return (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);
}
// Lane `from`'s value (`from` the same in every lane).
__device__ __forceinline__ uint32_t lane_value(uint32_t v, uint32_t from) {
  return uint32_t(__builtin_amdgcn_readlane(int(v), int(__builtin_amdgcn_readfirstlane(int(from)))));
}
__device__ __forceinline__ float lane_value(float v, uint32_t from) { return __uint_as_float(lane_value(__float_as_uint(v), from)); }
// A row's sixteen values in candidate order, summed in that order.
__device__ __forceinline__ float ordered_sum(const float *values) {
  float sum = 0.f;
#pragma unroll
  for (uint32_t c = 0; c < kCandidates; ++c) sum += values[c];
  return sum;
}

// By position, predecessor and candidate: the draft's probability, the lane's tempered one, and its estimate.
struct TreeState {
  float probability[kPositions][kCandidates][kCandidates];
  float drafted[kPositions][kCandidates][kCandidates];
  float logDrafted[kPositions][kCandidates][kCandidates];
  float estimate[kPositions][kCandidates][kCandidates];
  uint32_t order[kPositions][kCandidates][kCandidates];
  uint8_t likeliest[kPositions][kCandidates][kChildren];
  uint32_t ids[kPositions][kCandidates];
};

} // namespace

constexpr uint32_t kTreeThreads = 1024, kLatticeThreads = kCandidates * kCandidates, kTeams = kTreeThreads / kLatticeThreads;
__global__ __launch_bounds__(kTreeThreads) void draft_select_tree(const uint32_t *__restrict__ candidates, const float *__restrict__ unary,
                                                         const float *__restrict__ edges, const uint32_t *__restrict__ chain_tokens,
                                                         const float *__restrict__ chain_rates, uint32_t *__restrict__ tokens,
                                                         AttentionTreeRow *__restrict__ tree, float *__restrict__ scores,
                                                         uint32_t *__restrict__ sizes, uint8_t *__restrict__ draws,
                                                         float *__restrict__ next, float *__restrict__ caps, DraftTreeParams p) {
  __shared__ TreeState s;
  const uint32_t lane = blockIdx.x, tid = threadIdx.x, i = tid & 15u;
  const size_t origin = size_t(lane) * kPositions * kCandidates;
  const float temperature = p.temperature[lane], slope = p.slope[lane];
  const uint32_t chain = tid < DRAFT_CHAIN_TOKENS ? chain_tokens[size_t(lane) * DRAFT_CHAIN_TOKENS + tid] : 0u;
  constexpr uint32_t kRates = DRAFT_CHAIN_TOKENS * DRAFT_CHAIN_AGREEMENTS;
  const float rates = tid < kRates ? chain_rates[size_t(lane) * kRates + tid] : 0.f;

  // ---- The lattice: sixteen threads, a candidate each, a predecessor (position 0 follows the anchor alone, predecessor 0;
  // what the others compute there is not read); a team of 256 threads every fourth position, its two side by side (one team,
  // seven positions a thread, took the longer half of the kernel; a launch of fewer threads has its teams' work done in
  // turns). Sixteen threads share a wavefront, whose LDS operations are in order, so nothing here waits for the workgroup.
  auto lattice = [&](uint32_t team) __attribute__((always_inline)) {
    constexpr uint32_t kEach = (kPositions + kTeams - 1u) / kTeams;
    const uint32_t predecessor = tid % kLatticeThreads / kCandidates;
    uint32_t positions[kEach];   // (one past the last: not worked, by whole wavefronts)
    float score[kEach], weight[kEach];
#pragma unroll
    for (uint32_t e = 0; e < kEach; ++e) {
      const uint32_t position = positions[e] = team + kTeams * e;
      if (position >= kPositions) break;
      const size_t at = origin + position * kCandidates;
      if (predecessor == 0) s.ids[position][i] = candidates[at + i];
      score[e] = unary[at + i] + edges[(at + predecessor) * kCandidates + i];
    }
    auto largest = [](float v) {   // of sixteen, as fmaxf has it
      v = fmaxf(v, __uint_as_float(dpp_move<kQuadSwap1>(__float_as_uint(v))));
      v = fmaxf(v, __uint_as_float(dpp_move<kQuadSwap2>(__float_as_uint(v))));
      v = fmaxf(v, __uint_as_float(dpp_move<kRowHalfMirror>(__float_as_uint(v))));
      return fmaxf(v, __uint_as_float(dpp_move<kRowMirror>(__float_as_uint(v))));
    };
#pragma unroll
    for (uint32_t e = 0; e < kEach; ++e) {
      const uint32_t position = positions[e];
      if (position >= kPositions) break;
      weight[e] = expf(score[e] - largest(score[e]));
      s.probability[position][predecessor][i] = weight[e];
      s.order[position][predecessor][i] = order_bits(score[e] + 0.0f);
    }
    wave_lds_fence();
#pragma unroll
    for (uint32_t e = 0; e < kEach; ++e) {
      const uint32_t position = positions[e];
      if (position >= kPositions) break;
      // the four likeliest, the lower index first among equal scores
      uint32_t rank = 0;
      const uint32_t mine = order_bits(score[e] + 0.0f);
#pragma unroll
      for (uint32_t c = 0; c < kCandidates; ++c) {
        const uint32_t other = s.order[position][predecessor][c];
        rank += other > mine || (other == mine && c < i) ? 1u : 0u;
      }
      if (rank < kChildren) s.likeliest[position][predecessor][rank] = uint8_t(i);
      weight[e] /= ordered_sum(s.probability[position][predecessor]);
    }
    wave_lds_fence();
#pragma unroll
    for (uint32_t e = 0; e < kEach; ++e) {
      const uint32_t position = positions[e];
      if (position >= kPositions) break;
      const float q = weight[e], top = largest(q);
      s.probability[position][predecessor][i] = q;
      weight[e] = temperature == 0.0f || !(q > 0.0f) ? q : expf((logf(q) - logf(top)) / temperature);
      s.drafted[position][predecessor][i] = weight[e];
    }
    wave_lds_fence();
#pragma unroll
    for (uint32_t e = 0; e < kEach; ++e)
      if (positions[e] < kPositions) weight[e] /= ordered_sum(s.drafted[positions[e]][predecessor]);
    wave_lds_fence();
#pragma unroll
    for (uint32_t e = 0; e < kEach; ++e) {
      const uint32_t position = positions[e];
      if (position >= kPositions) break;
      s.drafted[position][predecessor][i] = weight[e];
      s.logDrafted[position][predecessor][i] = logf(weight[e]);
      const float q = fminf(fmaxf(weight[e], 1.0e-6f), 1.0f - 1.0e-6f);
      const float z = slope * logf(q / (1.0f - q)) + p.intercept[lane][position];
      s.estimate[position][predecessor][i] = 1.0f / (1.0f + expf(-z));
    }
  };
  lattice(tid / kLatticeThreads);
  if (__builtin_expect(blockDim.x < kTreeThreads, 0))
    for (uint32_t team = tid / kLatticeThreads + max(1u, blockDim.x / kLatticeThreads); team < kTeams; team += max(1u, blockDim.x / kLatticeThreads))
      lattice(team);
  __syncthreads();
  if (tid >= 64u) return;

  // ---- The growth, by the first wavefront. Thread r holds row r, thread e open entry e (and 64 + e).
  const uint32_t children = min(p.children[lane], kChildren), deepest = p.depth[lane], chained = min(p.chain[lane], uint32_t(DRAFT_CHAIN_TOKENS));
  static_assert(kRates <= 64 && kRows <= 64 && kEntries <= 128 && kChildren == 4, "a thread a rate, a row, two entries; four draws a word");
  uint32_t made = 1, entryCount = 0, expanded = 0;
  uint32_t rowToken = p.anchor[lane], rowAncestors = 1u, rowParent = SAMPLING_TREE_ROOT, rowDepth = 0, rowOnChain = 1u, rowPredecessor = 0;
  uint32_t rowDraws = SAMPLING_NO_DRAW * 0x01010101u;
  uint32_t rowKeyLow = p.noise[lane][0], rowKeyHigh = p.noise[lane][1];
  float rowQ = 1.0f, rowEstimate = 1.0f, rowCap = 1.0f, rowLeft[kChildren] = {};
  uint64_t entryKey[2] = {0, 0};   // 0: taken, or none
  uint32_t entryInfo[2] = {0, 0};
  float entryScore[2] = {0.f, 0.f};

  // A host chain token's rate at depth d, by its agreement with the draft there: its likeliest candidate, another of its
  // candidates, none of them, or past its positions.
  auto chainRate = [&](uint32_t d) __attribute__((always_inline)) {
    const uint32_t token = lane_value(chain, d);
    uint32_t agreement = 3;
    if (d < kPositions) {
      const bool mine = tid < kCandidates && s.ids[d][i] == token;
      const uint64_t among = __builtin_amdgcn_ballot_w64(mine);
      agreement = among & 1u ? 0u : among ? 1u : 2u;
    }
    return lane_value(rates, d * DRAFT_CHAIN_AGREEMENTS + agreement);
  };
  auto push = [&](float score, uint32_t info) __attribute__((always_inline)) {
    if (entryCount >= kEntries) return;
    const uint64_t key = uint64_t(order_bits(score + 0.0f)) << 32 | (kDead - entryCount);
#pragma unroll
    for (uint32_t half = 0; half < 2; ++half)
      if (tid + 64u * half == entryCount) {
        entryKey[half] = key;
        entryInfo[half] = info;
        entryScore[half] = score;
      }
    ++entryCount;
  };
  auto capOf = [&](uint32_t parent, uint32_t index) __attribute__((always_inline)) {
    const uint32_t drawn = lane_value(rowDraws, parent);
    float cap = 1.0f;
#pragma unroll
    for (uint32_t child = kChildren; child-- > 0;)
      if ((drawn >> (8u * child) & 0xFFu) == index) cap = lane_value(rowLeft[child], parent);
    return cap;
  };
  // A draft row's children at `position`, after its candidate `predecessor`: its drawn candidates, each an entry.
  auto expand = [&](uint32_t row, uint32_t position, uint32_t predecessor, float score, bool hasChain, uint32_t chainToken,
                    float chainRateHere) __attribute__((always_inline)) {
    const float q = s.probability[position][predecessor][i], mine = s.drafted[position][predecessor][i];
    const float estimate = s.estimate[position][predecessor][i];
    const float logMine = s.logDrafted[position][predecessor][i];
    const uint32_t id = s.ids[position][i], likeliest = *reinterpret_cast<const uint32_t *>(s.likeliest[position][predecessor]);
    if (tid < kCandidates) next[(size_t(lane) * kRows + row) * kCandidates + i] = mine;
    expanded |= 1u << row;
    if (tid == row) rowPredecessor = predecessor;
    float key = -INFINITY;
    if (temperature > 0.0f) {
      const uint64_t rowKey = uint64_t(lane_value(rowKeyHigh, row)) << 32 | lane_value(rowKeyLow, row);
      if (mine > 0.0f) key = logMine + gumbel_of(rowKey, id);
    }
    uint32_t taken = 0;
    float bound = score, left = 1.0f - chainRateHere, reserved = chainRateHere;
#pragma unroll
    for (uint32_t child = 0; child < kChildren; ++child) {
      if (child >= children) break;
      uint32_t drawn = kCandidates;
      if (temperature == 0.0f) {
        const uint32_t likely = uint32_t(__builtin_amdgcn_readfirstlane(int(likeliest))) >> (8u * child) & 0xFFu;
        drawn = lane_value(q, likely) > 0.0f ? likely : kCandidates;
      } else {
        const uint32_t open = !(taken >> i & 1u) && key > -INFINITY ? order_bits(key) : 0u;
        const uint32_t best = row_max_dpp(open);
        const uint64_t at = __builtin_amdgcn_ballot_w64(open && open == best);
        drawn = at ? uint32_t(__builtin_ctzll(at)) : kCandidates;   // (the sixteen lanes four times over)
      }
      if (drawn == kCandidates) break;
      taken |= 1u << drawn;
      const bool joins = hasChain && lane_value(id, drawn) == chainToken;
      const float cap = joins ? left + reserved : left;
      const float own = fminf(lane_value(estimate, drawn), cap);
      left = joins ? cap - fmaxf(own, reserved) : left - own;
      reserved = joins ? 0.0f : reserved;
      bound = fminf(bound, score * own);
      if (tid == row) {
        rowDraws = (rowDraws & ~(0xFFu << (8u * child))) | drawn << (8u * child);
        rowLeft[child] = cap;
      }
      push(bound, row << 16 | position << 8 | drawn);
    }
  };

  if (deepest > 0) {
    const float rate = chained ? chainRate(0) : 0.0f;
    expand(0, 0, 0, 1.0f, chained != 0, chained ? lane_value(chain, 0) : 0u, rate);
    if (chained) push(rate, kChainEntry);
  }
  const uint32_t most = min(kRows, deepest + 1u);
  while (made < most) {
    // the best open entry: the largest estimate, the earliest made among equal ones
    const uint64_t best = wave_max_dpp(entryKey[0] > entryKey[1] ? entryKey[0] : entryKey[1]);
    if (!best) break;
    const uint32_t entry = kDead - uint32_t(best);
    const float score = lane_value(entry < 64u ? entryScore[0] : entryScore[1], entry & 63u);
    const uint32_t info = lane_value(entry < 64u ? entryInfo[0] : entryInfo[1], entry & 63u);
#pragma unroll
    for (uint32_t half = 0; half < 2; ++half)
      if (tid + 64u * half == entry) entryKey[half] = 0;
    const bool fromChain = (info & kChainEntry) != 0;
    const uint32_t parent = info >> 16 & 0x7FFFu, position = info >> 8 & 0xFFu, index = info & 0xFFu;
    const uint32_t drafted = min(position, kPositions - 1u);   // (a chain step's position may lie past the draft's)
    const uint32_t id = uint32_t(__builtin_amdgcn_readfirstlane(int(s.ids[drafted][index & 15u]))), token = fromChain ? lane_value(chain, position) : id;
    // (a draft step's own probability: in the distribution its parent's children were drawn from)
    const float q = fromChain ? -1.0f : s.drafted[drafted][lane_value(rowPredecessor, parent)][index & 15u];
    // a token path the tree holds already gains no row
    const uint64_t same = __builtin_amdgcn_ballot_w64(tid >= 1u && tid < made && rowParent == parent && rowToken == token);
    uint32_t row = same ? uint32_t(__builtin_ctzll(same)) : 0u;
    if (!row) {
      row = made++;
      const float cap = fromChain ? 1.0f : capOf(parent, index);
      const uint32_t ancestors = lane_value(rowAncestors, parent);
      const bool onChain = lane_value(rowOnChain, parent) && position < chained && token == lane_value(chain, position);
      const uint64_t parentKey = uint64_t(lane_value(rowKeyHigh, parent)) << 32 | lane_value(rowKeyLow, parent);
      const uint64_t key = mix64(parentKey + 0x9e3779b97f4a7c15ull * (uint64_t(token) + 1u));
      if (tid == row) {
        rowToken = token;
        rowAncestors = ancestors | 1u << row;
        rowParent = parent;
        rowDepth = position + 1u;
        rowOnChain = onChain;
        rowQ = q;   // (a row a host chain token made is no draft step)
        rowEstimate = score;
        rowCap = cap;
        rowKeyLow = uint32_t(key);
        rowKeyHigh = uint32_t(key >> 32);
      }
    } else if (!fromChain && lane_value(rowQ, row) < 0.0f) {
      // a draft step that joins a host chain's row gives it its draft probability and cap
      const float cap = capOf(parent, index);
      if (tid == row) {
        rowQ = q;
        rowCap = cap;
      }
    }
    if (position + 1u >= deepest) continue;   // the row's children would lie too deep
    const bool chainChild = lane_value(rowOnChain, row) && position + 1u < chained;
    if (!fromChain && position + 1u < kPositions)
      expand(row, position + 1u, index, score, chainChild, chainChild ? lane_value(chain, position + 1u) : 0u, chainChild ? chainRate(position + 1u) : 0.0f);
    else if (fromChain && position + 1u < chained)
      push(score * chainRate(position + 1u), kChainEntry | row << 16 | (position + 1u) << 8);
  }
  if (tid == 0) sizes[lane] = made;
  if (tid < made) {
    const size_t at = size_t(lane) * kRows + tid;
    tokens[at] = rowToken;
    tree[at] = AttentionTreeRow{rowAncestors, uint16_t(rowParent), uint16_t(rowDepth)};
    scores[2 * at] = rowQ;
    scores[2 * at + 1] = rowEstimate;
    caps[at] = rowCap;
#pragma unroll
    for (uint32_t child = 0; child < kChildren; ++child) draws[at * kChildren + child] = uint8_t(rowDraws >> (8u * child));
  }
  for (uint32_t k = tid; k < made * kCandidates; k += 64u)   // (a row that was expanded has its probabilities already)
    if (!(expanded >> (k / kCandidates) & 1u)) next[size_t(lane) * kRows * kCandidates + k] = 0.f;
}
SP_REGISTER_KERNEL("draft_select_tree", &draft_select_tree);

// The trees' side of a sampled verify step, gathered by the step's rows (abi/Sampling.h, VerifyChildrenParams).
__global__ __launch_bounds__(64) void draft_verify_children(const uint32_t *__restrict__ sources, const SamplingLaneRows *__restrict__ lane_rows,
                                                            const AttentionTreeRow *__restrict__ step_tree, const uint32_t *__restrict__ candidates,
                                                            const float *__restrict__ tree_next, const uint8_t *__restrict__ tree_draws,
                                                            uint32_t *__restrict__ ids, float *__restrict__ probabilities,
                                                            uint8_t *__restrict__ draws, uint32_t *__restrict__ depths, VerifyChildrenParams p) {
  const uint32_t row = blockIdx.x, tid = threadIdx.x;
  if (row >= p.rows) return;
  uint32_t lane = SAMPLING_MAXIMUM_LANES;
  for (uint32_t l = 0; l < min(p.lanes, uint32_t(SAMPLING_MAXIMUM_LANES)); ++l)
    if (row >= lane_rows[l].first && row < lane_rows[l].first + lane_rows[l].rows) lane = l;
  const uint32_t source = sources[row], depth = step_tree[row].depth;
  const bool drafted = lane < SAMPLING_MAXIMUM_LANES && source < kRows && depth < kPositions;
  if (tid == 0) depths[row] = lane < SAMPLING_MAXIMUM_LANES ? depth : 0u;
  if (tid < kCandidates) {
    ids[size_t(row) * kCandidates + tid] = drafted ? candidates[(size_t(lane) * kPositions + depth) * kCandidates + tid] : SAMPLING_NO_TOKEN;
    probabilities[size_t(row) * kCandidates + tid] = drafted ? tree_next[(size_t(lane) * kRows + source) * kCandidates + tid] : 0.f;
  }
  if (tid < kChildren) draws[size_t(row) * kChildren + tid] = drafted ? tree_draws[(size_t(lane) * kRows + source) * kChildren + tid] : uint8_t(SAMPLING_NO_DRAW);
}
SP_REGISTER_KERNEL("draft_verify_children", &draft_verify_children);

} // namespace splash::kernels
