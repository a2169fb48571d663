// rans_bound.hip -- the most bytes that a reference rANS segment of n symbols
// can shed (ptwm_amd/csrc/ref_rans.h), on the host: before each symbol any
// state meets any thresholds, then identity steps follow from any state.
#include <algorithm>
#include <random>

#include "ref_rans.h"

using namespace ptwm;

// 0 if no run of n symbols and `tail` identity steps passes the scratch
// (x_final and the shed bytes), else the bytes past it.
extern "C" uint64_t rans_bound(uint64_t n, uint32_t tail, uint32_t seed) {
  std::mt19937 rng(seed);
  const uint32_t edge[] = {0u, 1u << 23, 0x7FFFFFFFu, 0x80000000u, 0xFFFFFFFFu};
  uint64_t most = 0;
  for (uint32_t run = 0; run < 64; ++run) {
    uint64_t bytes = 4;
    for (uint64_t i = 0; i < n; ++i) {
      // the entry of a symbol that the counts did not hold has thresholds 0
      const uint32_t th = run & 1 ? 0u : (uint32_t)rng();
      bytes += shed(run < 32 ? 0xFFFFFFFFu : (uint32_t)rng(), th);
    }
    uint32_t x = run % 8 < 5 ? edge[run % 8] : (uint32_t)rng();
    for (uint32_t i = 0; i < tail; ++i) {
      const uint32_t k = shed(x, kRansIdentityTh);
      bytes += k;
      x >>= 8 * k;
    }
    most = std::max(most, bytes);
  }
  const uint64_t room = ref_rans_scratch(n);
  return most > room ? most - room : 0;
}

// Whether identity steps leave a state of the format (below 2^31) alone.
extern "C" int rans_identity(uint32_t x) { return shed(x, kRansIdentityTh) == 0; }
