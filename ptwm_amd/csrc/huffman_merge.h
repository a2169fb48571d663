// huffman_merge.h -- the choice of the two-queue Huffman merge's next step
// (code_tables.hip), apart so that it can be compiled and checked on the host.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ptwm {

constexpr uint32_t kMergeNone = 0xFFFFFFFFu;
constexpr uint32_t kMergeRound = 16;  // items that make a round worth its barriers (0.14 us a step, 1 us a round)

// The two FIFO queues: leaves [li, n) in ascending order, internal nodes
// [qi, qe) in creation order, in which their counts never decrease.
struct MergeQueues {
  uint32_t li, qi, qe;
};

struct MergeStep {
  uint32_t both;        // the two smallest together
  bool a_leaf, b_leaf;  // what they are
  bool round;           // kMergeRound items or more of one queue are no larger than `both`
};

// leaf[n .. n + kMergeRound) is kMergeNone.  The wavefronts of a workgroup take
// the steps between two barriers each for itself, and one may be any number of
// steps behind another: entries of `node` from this wavefront's own qe on hold
// either what an earlier call left or what a wavefront ahead has stored, so
// they are read (the read costs the same either way) and not used.
__host__ __device__ inline MergeStep merge_step(const uint32_t* leaf, const uint32_t* node, const MergeQueues& m) {
  const uint32_t l0 = leaf[m.li], l1 = leaf[m.li + 1], l_far = leaf[m.li + kMergeRound - 1];
  const uint32_t n0 = node[m.qi], n1 = node[m.qi + 1], n_far = node[m.qi + kMergeRound - 1];
  const uint32_t queued = m.qe - m.qi;
  const uint32_t i0 = queued > 0 ? n0 : kMergeNone, i1 = queued > 1 ? n1 : kMergeNone;
  const uint32_t i_far = queued >= kMergeRound ? n_far : kMergeNone;
  MergeStep s;
  s.a_leaf = l0 <= i0;
  s.b_leaf = s.a_leaf ? l1 <= i0 : l0 <= i1;
  s.both = (s.a_leaf ? l0 : i0) + (s.b_leaf ? (s.a_leaf ? l1 : l0) : (s.a_leaf ? i0 : i1));
  s.round = l_far <= s.both || i_far <= s.both;
  return s;
}

// The queues after a step of one pair (the pair's parent is node m.qe).
__host__ __device__ inline MergeQueues merge_next(const MergeQueues& m, const MergeStep& s) {
  const uint32_t leaves = (s.a_leaf ? 1u : 0u) + (s.b_leaf ? 1u : 0u);
  return MergeQueues{m.li + leaves, m.qi + 2u - leaves, m.qe + 1u};
}

}  // namespace ptwm
