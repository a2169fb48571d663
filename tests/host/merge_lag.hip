// merge_lag.hip -- the Huffman table build's serial merge as the four
// wavefronts of a workgroup take it between barriers, on the host: each steps
// for itself (ptwm_amd/csrc/huffman_merge.h) on shared arrays, in a given
// schedule.
#include <algorithm>
#include <random>
#include <vector>

#include "huffman_merge.h"

using namespace ptwm;

// count[0..n) ascending, n >= 2.  lag 0: wavefront 0 runs ahead as far as it
// can, then the next; else a random schedule of that seed.  fill: what `node`
// holds before.  depth[i]: of leaf i.  0, or -1 when the wavefronts part.
extern "C" int merge_lag(const uint32_t* count, uint32_t n, uint32_t lag, uint32_t fill, uint32_t* depth) {
  constexpr uint32_t kWaves = 4;
  std::vector<uint32_t> leaf(256 + kMergeRound, kMergeNone), node(256 + kMergeRound, fill), up(512, 0);
  std::copy(count, count + n, leaf.begin());
  std::mt19937 rng(lag);
  MergeQueues m[kWaves] = {};
  auto live = [&](const MergeQueues& q) { return n - q.li + (q.qe - q.qi) > 1; };
  while (true) {
    bool waits[kWaves] = {}, rounds[kWaves] = {};
    for (uint32_t waiting = 0; waiting < kWaves;) {
      uint32_t w = 0;
      if (lag) w = rng() % kWaves;
      while (waits[w]) w = (w + 1) % kWaves;
      MergeQueues& q = m[w];
      const MergeStep s = live(q) ? merge_step(leaf.data(), node.data(), q) : MergeStep{};
      if (!live(q) || s.round) {
        rounds[w] = s.round;
        waits[w] = true;
        ++waiting;
        continue;
      }
      if (q.qe >= 255) return -1;
      const uint32_t a = s.a_leaf ? q.li : 256 + q.qi;
      const uint32_t b = s.b_leaf ? q.li + (s.a_leaf ? 1 : 0) : 256 + q.qi + (s.a_leaf ? 0 : 1);
      node[q.qe] = s.both;
      up[a] = up[b] = 256 + q.qe;
      q = merge_next(q, s);
    }
    for (uint32_t w = 1; w < kWaves; ++w)
      if (rounds[w] != rounds[0] || m[w].li != m[0].li || m[w].qi != m[0].qi || m[w].qe != m[0].qe) return -1;
    if (!rounds[0]) break;
    // a round: the items no larger than the first pair's sum, in order, in pairs
    MergeQueues q = m[0];
    const uint32_t both = merge_step(leaf.data(), node.data(), q).both;
    std::vector<uint32_t> items;
    uint32_t li = q.li, qi = q.qi;
    while (true) {
      const bool l = li < n && leaf[li] <= both, i = qi < q.qe && node[qi] <= both;
      if (!l && !i) break;
      if (l && (!i || leaf[li] <= node[qi])) items.push_back(li++);
      else items.push_back(256 + qi++);
    }
    if (items.size() < 2) return -1;
    for (size_t k = 0; k + 1 < items.size(); k += 2) {
      uint32_t sum = 0;
      for (size_t j = k; j < k + 2; ++j) {
        const uint32_t id = items[j];
        sum += id < 256 ? leaf[id] : node[id - 256];
        up[id] = 256 + q.qe;
        id < 256 ? ++q.li : ++q.qi;
      }
      node[q.qe++] = sum;
    }
    std::fill(m, m + kWaves, q);
  }
  for (uint32_t i = 0; i < n; ++i) {
    depth[i] = 0;
    for (uint32_t id = i; id != 256 + n - 2; id = up[id])
      if (++depth[i] > 256) return -1;
  }
  return 0;
}
