// code_tables.hip -- canonical Huffman codes and rANS frequency tables from
// 256-bin histograms, one workgroup per table, a thread per symbol.
//
// The tables are the reference encoder's bit for bit (entropy/huffman/
// tree.rs:19-177, weights.rs:8-32, rans/compress.rs:35-122; huffman_host.cpp
// is the host form of the code lengths).  On the host a table took 6.6 us and
// the histograms had to be fetched and the codes sent back, with the device
// idle: 1.7 ms of a 5.6 ms call for the 256 chunk tables of a 64 MiB fp32
// tensor.  Here all tables of a call are built at once.
//
// The tree: leaves sorted by (count, symbol) by counting the smaller ones,
// then the two-queue merge, the only serial part: a step per symbol, four LDS
// reads that depend on the step before, 0.14 us each, run by all threads
// alike.  Where many items are no larger than the two smallest together, none
// of the nodes made of them can come before any of them, so they are paired
// all at once (a flat 256-symbol alphabet takes 5 such rounds and some 20
// steps instead of 255).  Depths by pointer jumping; the rest is a few ballots.
#include "code_tables.h"

#include "huffman_merge.h"
#include "ref_rans.h"

namespace ptwm {

namespace {

constexpr uint32_t kNone = kMergeNone;
constexpr uint32_t kScale = 2048;     // rANS frequencies sum to 2^11
constexpr uint32_t kThreads = 256;
constexpr uint32_t kRound = kMergeRound;

struct Scratch {
  u32x4 f4[64];                 // counts by symbol
  uint32_t leaf[256 + kRound];  // counts of the sorted leaves, then kNone
  uint32_t node[256 + kRound];  // counts of the internal nodes, in creation order
  uint32_t order[256];          // a round's counts in order
  uint16_t up[512];             // parent: leaf i at i, internal node q at 256 + q
  uint16_t dist[512];           // edges to `up`
  uint8_t sym[256];             // symbol of leaf i
  uint8_t len[256];             // code length by symbol
  uint32_t head[132];           // header bytes, 4-byte aligned
  uint32_t count[4][12];        // per wavefront: symbols of each length
  uint64_t part[4];
};

// Sum, minimum and maximum over the workgroup (every thread calls).
__device__ __forceinline__ uint64_t sum_all(Scratch& S, uint64_t v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor((unsigned long long)v, d, 64);
  __syncthreads();
  if ((threadIdx.x & 63u) == 0) S.part[threadIdx.x >> 6] = v;
  __syncthreads();
  return S.part[0] + S.part[1] + S.part[2] + S.part[3];
}
__device__ __forceinline__ uint32_t min_all(Scratch& S, uint32_t v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = min(v, (uint32_t)__shfl_xor(v, d, 64));
  __syncthreads();
  if ((threadIdx.x & 63u) == 0) S.part[threadIdx.x >> 6] = v;
  __syncthreads();
  return (uint32_t)min(min(S.part[0], S.part[1]), min(S.part[2], S.part[3]));
}

// Items of the ascending list a[lo .. hi) below v (kEqual: or equal to it).
template <bool kEqual>
__device__ __forceinline__ uint32_t below(const uint32_t* a, uint32_t lo, uint32_t hi, uint32_t v) {
  const uint32_t lo0 = lo;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (kEqual ? a[mid] <= v : a[mid] < v) lo = mid + 1;
    else hi = mid;
  }
  return lo - lo0;
}

// Code length of symbol t (tree.rs:19-85, 212-242), its count h; n symbols
// have nonzero counts.
__device__ uint32_t huffman_length(Scratch& S, uint32_t h, uint32_t n, uint32_t max_len) {
  const uint32_t t = threadIdx.x;
  if (n == 1) return h ? 1u : 0u;
  reinterpret_cast<uint32_t*>(S.f4)[t] = h;
  for (uint32_t i = t; i < 256 + kRound; i += kThreads) S.leaf[i] = kNone;
  S.len[t] = 0;
  __syncthreads();
  // rank: symbols with (count, symbol) below this one's; a count of zero
  // wraps to the largest value
  uint32_t rank = 0;
#pragma unroll 4
  for (uint32_t j = 0; j < 64; ++j) {
    const u32x4 f = S.f4[j];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) rank += f[i] - 1u < h - 1u + (4 * j + i < t ? 1u : 0u) ? 1u : 0u;
  }
  if (h) {
    S.leaf[rank] = h;
    S.sym[rank] = (uint8_t)t;
  }
  __syncthreads();
  // Two FIFO queues: the sorted leaves and the internal nodes; a leaf goes
  // first on ties (its id is smaller).  Every thread takes every step: the
  // writes are alike, each thread uses only what it wrote itself since the
  // last barrier (merge_step), and so all wavefronts reach the same rounds and
  // the same end.  Counts of up to 2^32 - 1 bytes in all stay below kNone
  // until the last pair.
  MergeQueues m{0, 0, 0};
  while (n - m.li + (m.qe - m.qi) > 1) {
    const MergeStep step = merge_step(S.leaf, S.node, m);
    const uint32_t li = m.li, qi = m.qi, qe = m.qe, both = step.both;
    if (step.round) {
      // a round: the items no larger than `both`, in order, in pairs; an odd
      // last one stays
      __syncthreads();  // (every wavefront has made its steps before)
      const uint32_t cl = below<true>(S.leaf, li, n, both), ci = below<true>(S.node, qi, qe, both);
      const uint32_t pairs = (cl + ci) / 2;
      if (t < cl) {
        const uint32_t f = S.leaf[li + t], r = t + below<false>(S.node, qi, qi + ci, f);
        S.order[r & 255u] = f;
        if (r < 2 * pairs) S.up[li + t] = (uint16_t)(256u + qe + r / 2);
      }
      if (t < ci) {
        const uint32_t f = S.node[qi + t], r = t + below<true>(S.leaf, li, li + cl, f);
        S.order[r & 255u] = f;
        if (r < 2 * pairs) S.up[256u + qi + t] = (uint16_t)(256u + qe + r / 2);
      }
      const bool odd = (cl + ci) & 1u;
      const bool last_leaf = cl && (!ci || S.leaf[li + cl - 1] > S.node[qi + ci - 1]);
      __syncthreads();
      if (t < pairs) S.node[qe + t] = S.order[2 * t] + S.order[2 * t + 1];
      m.li += cl - (odd && last_leaf ? 1u : 0u);
      m.qi += ci - (odd && !last_leaf ? 1u : 0u);
      m.qe += pairs;
      __syncthreads();
      continue;
    }
    const uint32_t a = step.a_leaf ? li : 256u + qi;
    const uint32_t b = step.b_leaf ? li + (step.a_leaf ? 1u : 0u) : 256u + qi + (step.a_leaf ? 0u : 1u);
    S.node[qe] = both;
    S.up[a] = S.up[b] = (uint16_t)(256u + qe);
    m = merge_next(m, step);
  }
  const uint32_t root = 256u + n - 2u;
  __syncthreads();
  // depths: every node's pointer jumps to its pointer's, distances add
  // (thread t: leaf t and internal node t)
  uint32_t up[2], d[2];
#pragma unroll
  for (uint32_t k = 0; k < 2; ++k) {
    const uint32_t id = t + 256 * k;
    const bool live = k == 0 ? t < n : id < root;
    up[k] = live ? S.up[id] : root;
    d[k] = live ? 1u : 0u;
  }
  for (;;) {
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) {
      S.up[t + 256 * k] = (uint16_t)up[k];
      S.dist[t + 256 * k] = (uint16_t)d[k];
    }
    if (!__syncthreads_or(up[0] != root)) break;  // (the leaves are the deepest)
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k)
      if (up[k] != root) {
        d[k] += S.dist[up[k]];
        up[k] = S.up[up[k]];
      }
  }
  // lengths, limited: Kraft's sum brought back by lengthening the shortest
  // code below the limit (its smallest symbol) until it fits
  const bool over = t < n && d[0] > max_len;
  if (t < n) S.len[S.sym[t]] = (uint8_t)min(d[0], max_len);
  const bool clamped = __syncthreads_or(over);
  uint32_t l = S.len[t];
  if (!clamped) return l;
  for (;;) {
    const uint32_t kraft = (uint32_t)sum_all(S, l ? 1u << (max_len - l) : 0u);
    const uint32_t best = min_all(S, l && l < max_len ? l << 8 | t : kNone);
    if (kraft <= 1u << max_len || best == kNone) return l;
    if ((best & 255u) == t) ++l;
  }
}

// Canonical bit-reversed code of symbol t (tree.rs:102-177); false if the
// lengths form no code.
__device__ bool canonical(Scratch& S, uint32_t l, uint32_t& rev) {
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  uint32_t rank = 0;
#pragma unroll
  for (uint32_t b = 1; b <= 11; ++b) {
    const uint64_t m = __ballot(l == b);
    if (l == b) rank = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) S.count[wave][b] = (uint32_t)__popcll(m);
  }
  __syncthreads();
  uint32_t code = 0, prev = 0;
  bool ok = true;
  rev = 0;
#pragma unroll
  for (uint32_t b = 1; b <= 11; ++b) {
    const uint32_t count = S.count[0][b] + S.count[1][b] + S.count[2][b] + S.count[3][b];
    code = (code + prev) << 1;  // first code of length b
    // (past the longest length the reference does not look)
    if (count && code + count > (1u << b)) ok = false;
    if (l == b) {
      uint32_t c = code + rank;
      for (uint32_t w = 0; w < wave; ++w) c += S.count[w][b];
      rev = __builtin_bitreverse32(c) >> (32u - b);
    }
    prev = count;
  }
  return ok;
}

__global__ void __launch_bounds__(kThreads) code_tables_kernel(const TableJob* __restrict__ jobs,
                                                               const uint32_t* __restrict__ hist,
                                                               uint32_t* __restrict__ codes, uint4* __restrict__ rans,
                                                               TableInfo* __restrict__ info) {
  __shared__ Scratch S;
  const uint32_t j = blockIdx.x, t = threadIdx.x;
  const TableJob J = jobs[j];
  TableInfo& I = info[j];
  const uint64_t at = reinterpret_cast<uint64_t>(hist + 256ull * J.row0 + t);
  uint32_t row[4] = {0, 0, 0, 0}, h = 0;
#pragma unroll
  for (uint32_t r = 0; r < 4; ++r) {
    if (r < J.rows) row[r] = g_ld<uint32_t>(at + 1024ull * r);
    h += row[r];
  }
  for (uint32_t i = t; i < 132; i += kThreads) S.head[i] = 0;
  const uint32_t n = (uint32_t)__syncthreads_count(h != 0);
  const uint32_t n_sym = 256u - min_all(S, h ? 255u - t : 256u);
  uint8_t* const head = reinterpret_cast<uint8_t*>(S.head);
  bool ok = n != 0;
  uint32_t head_len = 0;
  if (ok && J.kind <= kTableIlv) {
    uint32_t rev;
    const uint32_t l = huffman_length(S, h, n, J.kind == kTableIlv && n_sym <= 16 ? 6u : 11u);
    ok = canonical(S, l, rev);
    g_st<uint32_t>(reinterpret_cast<uint64_t>(codes + 256ull * j + t), l << 16 | rev);
    // weights header: 0x80 | count, or 0x80 and count (256 as 0), then the
    // lengths, two to a byte
    const uint32_t hb = n_sym <= 127 ? 1u : 2u;
    head_len = hb + (n_sym + 1) / 2;
    if (t == 0) {
      head[0] = (uint8_t)(0x80u | (n_sym <= 127 ? n_sym : 0u));
      if (hb == 2) head[1] = (uint8_t)n_sym;
    }
    const uint32_t next = __shfl_down(l, 1, 64);
    if (!(t & 1u) && t < n_sym) head[hb + t / 2] = (uint8_t)(l | next << 4);
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
      if (r >= J.rows) break;
      const uint64_t bits = sum_all(S, (uint64_t)row[r] * l);
      if (t == 0) I.bits[r] = bits;
    }
  } else if (ok) {
    // normalize_freqs (rans/compress.rs:72-122); the first symbol with the
    // largest count takes the rounding
    const uint64_t total = sum_all(S, h);
    uint32_t f = h ? max((uint32_t)((uint64_t)h * kScale / total), 1u) : 0u;
    const uint32_t assigned = (uint32_t)sum_all(S, f);
    const uint32_t most = kNone - min_all(S, kNone - h);
    const uint32_t first = min_all(S, h == most ? t : kNone);
    const bool refused = t == first && assigned > kScale && f <= assigned - kScale;
    if (t == first) f += kScale - assigned;
    ok = !__syncthreads_or(refused);
    if (ok) {
      uint32_t incl = f;
#pragma unroll
      for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(incl, d, 64);
        if ((t & 63u) >= d) incl += o;
      }
      if ((t & 63u) == 63u) S.count[t >> 6][0] = incl;
      __syncthreads();
      uint32_t start = incl - f;
      for (uint32_t w = 0; w < t >> 6; ++w) start += S.count[w][0];
      if (t >= n_sym) start = 0;
      if (J.kind == kTableRansIlv) {
        codes[256ull * j + t] = f | start << 16;
        const double gain = 11.0 - log2((double)max(f, 1u)) - 2.25e-5 * f;  // rans_ilv_least
        const uint64_t bits = sum_all(S, (uint64_t)((double)h * (gain > 0 ? gain : 0)));
        if (t == 0) I.bits[0] = bits;
      } else {
        // EncSymbol (rans/compress.rs:35-68): {rcp, bias, cmpl | shift << 24},
        // and the thresholds that shed takes (ref_rans.h)
        uint4 e;
        if (f < 2) {
          e = make_uint4(kNone, start + kScale - 1, kScale - f, 0u);
        } else {
          const uint32_t sh = 32u - (uint32_t)__builtin_clz(f - 1u);  // 2^sh >= f
          const uint32_t rcp = (uint32_t)(((1ull << (sh + 31)) + f - 1) / f);
          e = make_uint4(rcp, start, (kScale - f) | (sh - 1) << 24, 0u);
        }
        if (f) e.w = ((f << 4) - 1u) | ((min(f, 8u) << 12) - 1u) << 16;
        rans[256ull * j + t] = e;
      }
      if (t < n_sym) {
        head[1 + 2 * t] = (uint8_t)f;
        head[2 + 2 * t] = (uint8_t)(f >> 8);
      }
      if (t == 0) head[0] = (uint8_t)(n_sym - 1);
      head_len = 1 + 2 * n_sym;
    } else if (J.kind == kTableRans) {
      // refused: the encoder, which runs before the host knows, goes over the
      // plane with entries that leave its state alone
      rans[256ull * j + t] = make_uint4(0u, 0u, 0u, kRansIdentityTh);
    }
  }
  __syncthreads();
  uint32_t* const out = reinterpret_cast<uint32_t*>(I.head);
  for (uint32_t i = t; 4 * i < head_len; i += kThreads) out[i] = S.head[i];
  if (t == 0) {
    I.ok = ok ? 1u : 0u;
    I.n_sym = n_sym;
    I.head_len = head_len;
  }
}

}  // namespace

hipError_t launch_code_tables(const TableJob* jobs, uint32_t n, const uint32_t* hist, uint32_t* codes, uint4* rans,
                              TableInfo* info, hipStream_t stream) {
  if (!n) return hipSuccess;
  hipLaunchKernelGGL(code_tables_kernel, dim3(n), dim3(kThreads), 0, stream, jobs, hist, codes, rans, info);
  return hipGetLastError();
}

}  // namespace ptwm
