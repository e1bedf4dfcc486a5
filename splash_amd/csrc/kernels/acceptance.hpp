// The greedy selection of a row and the acceptance of a lane's block, shared by the kernels of sampling.hip and the
// commit of paged_attention.hip that accepts its block itself.
#pragma once
#include "abi/PagedAttention.h"
#include "abi/Sampling.h"
#include "kernels/device_common.hpp"

namespace splash::kernels {

__device__ __forceinline__ bool unselectable(float v) { return !(v > -INFINITY); }  // NaN or -inf (sampling.metal:986-989)

struct Best {
  float value;
  uint32_t index;
};
__device__ __forceinline__ Best better(Best a, Best b) {
  return (b.value > a.value || (b.value == a.value && b.index < a.index)) ? b : a;
}
// The best of `Lanes` neighbouring lanes, in each of them.
template <int Lanes = 64> __device__ __forceinline__ Best wave_best(Best v) {
  if constexpr (Lanes > 32) v = better(v, Best{lane_xor<32>(v.value), lane_xor<32>(v.index)});
  if constexpr (Lanes > 16) v = better(v, Best{lane_xor<16>(v.value), lane_xor<16>(v.index)});
  if constexpr (Lanes > 8) v = better(v, Best{lane_xor<8>(v.value), lane_xor<8>(v.index)});
  if constexpr (Lanes > 4) v = better(v, Best{lane_xor<4>(v.value), lane_xor<4>(v.index)});
  if constexpr (Lanes > 2) v = better(v, Best{lane_xor<2>(v.value), lane_xor<2>(v.index)});
  if constexpr (Lanes > 1) v = better(v, Best{lane_xor<1>(v.value), lane_xor<1>(v.index)});
  return v;
}

// What sampling.metal:2044-2083 decides of a lane's block, by one wavefront, a thread a row (thread `row`, `live` below
// the lane's rows): a row follows its parent when its input token is the parent's selection and no earlier row of the
// same parent does (one ballot); a row lies on the accepted path when every row of its ancestor mask follows its parent.
// The path's rows, by depth, are the accepted draft tokens' rows; each selects the next token of the output, the last
// the target's own. The output is cut to what the lane may still keep and after its first stop token (a second ballot);
// the retained rows are the ancestor mask of the last kept row.
struct Acceptance {
  uint32_t kept, accepted;  // of the lane
  bool retains, last;       // the row's selection is output `depth`; it is the last one, whose ancestors are retained
  uint32_t depth;
};
__device__ __forceinline__ Acceptance accept_rows(uint32_t row, bool live, const AttentionTreeRow &node, uint32_t input,
                                                  uint32_t selection, uint32_t remaining, const uint32_t (&stopTokens)[SAMPLING_STOP_TOKENS]) {
  const uint32_t parent = live && row ? min(uint32_t(node.parent), SAMPLING_MAXIMUM_ROWS - 1u) : 0u;
  const uint32_t parentSelection = __shfl(selection, int(parent), 64);
  const bool matches = live && row && node.parent < row && input == parentSelection;
  // whether a matching row of this row's parent comes before it (each row's is the same word for the whole wavefront)
  const int matched = matches ? int(parent) : -1;
  bool follows = matches;
#pragma unroll
  for (uint32_t other = 1; other < SAMPLING_MAXIMUM_ROWS; ++other)
    if (__builtin_amdgcn_readlane(matched, int(other)) == int(parent) && other < row) follows = false;
  const uint32_t following = uint32_t(__builtin_amdgcn_ballot_w64(follows)) | 1u;   // the anchor starts the path
  const bool onPath = live && (node.ancestors & ~following) == 0u && ((node.ancestors >> row) & 1u);
  const uint32_t path = uint32_t(__builtin_amdgcn_ballot_w64(onPath));
  Acceptance a;
  a.accepted = uint32_t(__builtin_popcount(path)) - 1u;
  a.depth = live ? uint32_t(__builtin_popcount(path & ((1u << row) - 1u))) : 0u;   // the path's rows rise with depth
  a.kept = min(a.accepted + 1u, max(remaining, 1u));
  bool stop = false;
#pragma unroll
  for (int s = 0; s < int(SAMPLING_STOP_TOKENS); ++s) stop = stop || (stopTokens[s] != SAMPLING_NO_TOKEN && selection == stopTokens[s]);
  // the shallowest path row within the kept ones that selects a stop token ends the output
  const uint32_t stops = uint32_t(__builtin_amdgcn_ballot_w64(onPath && a.depth < a.kept && stop));
  if (stops) a.kept = uint32_t(__builtin_popcount(path & ((2u << __builtin_ctz(stops)) - 1u)));
  a.retains = onPath && a.depth < a.kept;
  a.last = onPath && a.depth + 1u == a.kept;
  a.accepted = min(a.accepted, a.kept);
  return a;
}

} // namespace splash::kernels
