// huffman_host.cpp -- Huffman code lengths on the host.
//
// The code lengths of the reference encoder (crates/ptwm-core/src/entropy/
// huffman/tree.rs:19-85, 212-242) from a 256-bin histogram, for the library's
// ptwm_mi355x_huffman_code_lengths; the encoders build their tables on the
// device (code_tables.hip, the same construction).
//
// Tie-breaking follows tree.rs:51-65: nodes are merged in ascending
// (frequency, id) order, leaves take ids 0..n-1 in ascending symbol order and
// internal nodes the following ids in creation order.  Internal frequencies
// never decrease in creation order, so two FIFO queues (sorted leaves,
// internal nodes) pop in exactly the order of the reference's binary heap.
#include "huffman_host.h"

#include <algorithm>
#include <cstring>

namespace ptwm {

bool huf_lengths_from_freqs(const uint32_t freqs[256], uint8_t lengths[256], int max_len) {
  if (max_len < 1 || max_len > kHufMaxBits) return false;
  std::memset(lengths, 0, 256);
  int sym[256];
  int n = 0;
  for (int i = 0; i < 256; ++i)
    if (freqs[i]) sym[n++] = i;
  if (n == 0) return false;
  if (n == 1) {
    lengths[sym[0]] = 1;
    return true;
  }
  // leaves sorted by (freq, id); ids are ascending symbol order already
  int order[256];
  for (int i = 0; i < n; ++i) order[i] = i;
  std::stable_sort(order, order + n, [&](int a, int b) { return freqs[sym[a]] < freqs[sym[b]]; });
  uint64_t f[512];
  int parent[512];
  for (int i = 0; i < n; ++i) f[i] = freqs[sym[i]];
  int li = 0;              // next leaf in `order`
  int qi = n, qe = n;      // internal-node FIFO [qi, qe)
  auto take = [&]() -> int {
    // pop the smaller (freq, id); leaves have smaller ids than internal nodes
    bool leaf_ok = li < n;
    bool int_ok = qi < qe;
    if (leaf_ok && (!int_ok || f[order[li]] <= f[qi])) return order[li++];
    return qi++;
  };
  while ((n - li) + (qe - qi) > 1) {
    int a = take();
    int b = take();
    f[qe] = f[a] + f[b];
    parent[a] = qe;
    parent[b] = qe;
    ++qe;
  }
  const int root = qe - 1;
  // depth = number of edges to the root (DFS in tree.rs:66-81 gives the same)
  int depth[512];
  depth[root] = 0;
  for (int id = root - 1; id >= 0; --id) {
    int d = depth[parent[id]] + 1;
    depth[id] = d > 255 ? 255 : d;
  }
  for (int i = 0; i < n; ++i) lengths[sym[i]] = (uint8_t)depth[i];
  // enforce_max_code_length (tree.rs:212-242)
  bool clamped = false;
  for (int s = 0; s < 256; ++s)
    if (lengths[s] > max_len) {
      lengths[s] = (uint8_t)max_len;
      clamped = true;
    }
  if (clamped) {
    const uint32_t cap = 1u << max_len;
    for (;;) {
      uint32_t kraft = 0;
      for (int s = 0; s < 256; ++s)
        if (lengths[s]) kraft += 1u << (max_len - lengths[s]);
      if (kraft <= cap) break;
      int victim = -1;
      for (int s = 0; s < 256; ++s)
        if (lengths[s] > 0 && lengths[s] < max_len && (victim < 0 || lengths[s] < lengths[victim])) victim = s;
      if (victim < 0) break;
      lengths[victim]++;
    }
  }
  return true;
}

}  // namespace ptwm

extern "C" int64_t ptwm_mi355x_huffman_code_lengths(const uint32_t* freqs, uint8_t* lengths_out) {
  if (!freqs || !lengths_out) return -1;
  return ptwm::huf_lengths_from_freqs(freqs, lengths_out) ? 0 : -1;
}
