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
// then the two-queue merge, the only serial part.  Its steps depend on each
// other, but none of the nodes made of the items that are no larger than the
// two smallest together can come before any of these items, so they are
// paired all at once: rounds of 0.3 us, by one wavefront, which needs no
// barriers for them.  (A step a pair, by four wavefronts with barriers around
// rounds of 16 items or more, took 0.22 us a pair: 29 of the 43 us of a
// 142-symbol table.)  Depths by pointer jumping; the rest is a few ballots.
#include "code_tables.h"

#include "ref_rans.h"

namespace ptwm {

namespace {

constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr uint32_t kScale = 2048;     // rANS frequencies sum to 2^11
constexpr uint32_t kThreads = 256;

struct Scratch {
  u32x4 f4[64];             // nonzero counts by symbol, then kNone
  uint32_t leaf[256 + 64];  // counts of the sorted leaves, then kNone
  uint32_t node[256 + 64];  // counts of the internal nodes, in creation order
  uint32_t order[128];      // a round's counts in order
  uint16_t up[512];         // parent: leaf i at i, internal node q at 256 + q
  uint16_t dist[512];       // edges to `up`
  uint8_t sym[256];         // symbol of leaf i
  uint8_t len[256];         // code length by symbol
  uint32_t head[132];       // header bytes, 4-byte aligned
  uint32_t count[4][16];    // per wavefront: symbols of each length
  uint64_t used[4];         // per wavefront: the symbols with nonzero counts
  uint64_t part[4];
};

// Over the wavefront, in lane 63 (all lanes active): rows of 16 by row shifts,
// then broadcasts of rows 0, 2 (to 1, 3) and of row 1 (to 2, 3).
template <uint32_t kCtrl, uint32_t kRows>
__device__ __forceinline__ uint32_t dpp(uint32_t old, uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, kCtrl, kRows, 0xF, false);
}
__device__ __forceinline__ uint32_t wave_sum63(uint32_t v) {
  v += dpp<0x111, 0xF>(0, v);
  v += dpp<0x112, 0xF>(0, v);
  v += dpp<0x114, 0xF>(0, v);
  v += dpp<0x118, 0xF>(0, v);
  v += dpp<0x142, 0xA>(0, v);
  return v + dpp<0x143, 0xC>(0, v);
}
__device__ __forceinline__ uint32_t wave_min63(uint32_t v) {
  v = min(v, dpp<0x111, 0xF>(kNone, v));
  v = min(v, dpp<0x112, 0xF>(kNone, v));
  v = min(v, dpp<0x114, 0xF>(kNone, v));
  v = min(v, dpp<0x118, 0xF>(kNone, v));
  v = min(v, dpp<0x142, 0xA>(kNone, v));
  return min(v, dpp<0x143, 0xC>(kNone, v));
}

// Sum (of values below 2^48) and minimum over the workgroup (every thread
// calls).
__device__ __forceinline__ uint64_t sum_all(Scratch& S, uint64_t v) {
  const uint32_t lo = wave_sum63((uint32_t)v & 0xFFFFFFu), hi = wave_sum63((uint32_t)(v >> 24));
  __syncthreads();
  if ((threadIdx.x & 63u) == 63u) S.part[threadIdx.x >> 6] = lo + ((uint64_t)hi << 24);
  __syncthreads();
  return S.part[0] + S.part[1] + S.part[2] + S.part[3];
}
__device__ __forceinline__ uint32_t min_all(Scratch& S, uint32_t v) {
  v = wave_min63(v);
  __syncthreads();
  if ((threadIdx.x & 63u) == 63u) S.part[threadIdx.x >> 6] = v;
  __syncthreads();
  return (uint32_t)min(min(S.part[0], S.part[1]), min(S.part[2], S.part[3]));
}

__device__ __forceinline__ uint32_t lane_of(uint32_t v, uint32_t lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane);
}

// What lanes of this wavefront wrote to LDS is there for its other lanes.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The two-queue merge of n >= 2 leaves, by one wavefront: S.up of all but the
// root.  Two FIFO queues: the sorted leaves [li, n) and the internal nodes
// [qi, qe), whose counts never decrease in creation order; a leaf goes first on
// ties (its id is smaller).  Each round takes up to 64 items of either queue.
// Counts of up to 2^32 - 1 bytes in all stay below kNone until the last pair.
__device__ __forceinline__ void merge_leaves(Scratch& S, uint32_t n) {
  const uint32_t lane = threadIdx.x;
  n = (uint32_t)__builtin_amdgcn_readfirstlane((int)n);
  uint32_t li = 0, qi = 0, qe = 0;
  while (n - li + (qe - qi) > 1) {
    const uint32_t nl = n - li, nq = qe - qi;
    const uint32_t a = S.leaf[li + lane], b = lane < nq ? S.node[qi + lane] : kNone;
    // the two smallest together, and the items no larger than that: the first
    // cl leaves and ci nodes
    const uint32_t l0 = lane_of(a, 0), l1 = lane_of(a, 1), i0 = lane_of(b, 0), i1 = lane_of(b, 1);
    const uint32_t both = min(min(__builtin_elementwise_add_sat(l0, l1), __builtin_elementwise_add_sat(l0, i0)),
                              __builtin_elementwise_add_sat(i0, i1));
    uint32_t cl = min((uint32_t)__popcll(__ballot(a <= both)), nl);
    uint32_t ci = min((uint32_t)__popcll(__ballot(b <= both)), nq);
    if (max(cl, ci) == 64) {  // more may follow: up to the last that surely goes before those
      const uint32_t al = cl == 64 ? lane_of(a, 63) : kNone, bl = ci == 64 ? lane_of(b, 63) : kNone;
      if (al <= bl) ci = (uint32_t)__popcll(__ballot(b < al));
      else cl = (uint32_t)__popcll(__ballot(a <= bl));
    }
    // their ranks among each other
    uint32_t ra = lane, rb = lane;
    const uint32_t both_kinds = cl ? ci : 0;
    for (uint32_t j0 = 0; j0 < both_kinds; j0 += 4)  // (past ci: larger than any of the leaves)
#pragma unroll
      for (uint32_t j = j0; j < j0 + 4; ++j) {
        const uint32_t v = lane_of(b, j);
        ra += a > v ? 1u : 0u;
        const uint32_t at = j + (uint32_t)__popcll(__ballot(a <= v));
        rb = lane == j ? at : rb;
      }
    // in pairs, in order; an odd last one stays, and gets its parent later
    const uint32_t items = cl + ci, pairs = items / 2, odd = items & 1u;
    if (lane < cl) {
      S.order[ra] = a;
      S.up[li + lane] = (uint16_t)(256u + qe + ra / 2);
    }
    if (lane < ci) {
      S.order[rb] = b;
      S.up[256u + qi + lane] = (uint16_t)(256u + qe + rb / 2);
    }
    wave_sync();
    const uint32_t sum = S.order[2 * lane] + S.order[2 * lane + 1];
    S.node[qe + lane] = sum;  // (what is past the pairs is not in the queue)
    wave_sync();
    const uint32_t odd_leaf = odd && lane_of(ra, (cl - 1) & 63u) == items - 1 ? 1u : 0u;
    li += cl - odd_leaf;
    qi += ci - (odd - odd_leaf);
    qe += pairs;
  }
}

// Code length of symbol t (tree.rs:19-85, 212-242), its count h; n symbols
// have nonzero counts, `below` of them come before t.
__device__ uint32_t huffman_length(Scratch& S, uint32_t h, uint32_t below, uint32_t n, uint32_t max_len) {
  const uint32_t t = threadIdx.x;
  if (n == 1) return h ? 1u : 0u;
  uint32_t* const counts = reinterpret_cast<uint32_t*>(S.f4);
  if (h) counts[below] = h;
  if (t >= n) counts[t] = kNone;
  for (uint32_t i = t; i < 256 + 64; i += kThreads) S.leaf[i] = kNone;
  S.len[t] = 0;
  __syncthreads();
  // rank: symbols with (count, symbol) below this one's
  uint32_t rank = 0;
#pragma unroll 8
  for (uint32_t j = 0; 4 * j < n; ++j) {
    const u32x4 f = S.f4[j];
    const uint32_t limit = h + (j < below / 4 ? 1u : 0u);
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) rank += f[i] < limit ? 1u : 0u;
  }
#pragma unroll
  for (uint32_t i = 0; i < 3; ++i) rank += i < below % 4 && S.f4[below / 4 & 63u][i] == h ? 1u : 0u;
  if (h) {
    S.leaf[rank] = h;
    S.sym[rank] = (uint8_t)t;
  }
  __syncthreads();
  if (t < 64) merge_leaves(S, n);
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
  uint32_t kraft = (uint32_t)sum_all(S, l ? 1u << (max_len - l) : 0u);
  while (kraft > 1u << max_len) {
    const uint32_t best = min_all(S, l && l < max_len ? l << 8 | t : kNone);
    if (best == kNone) break;
    if ((best & 255u) == t) ++l;
    kraft -= 1u << (max_len - 1u - (best >> 8));
  }
  return l;
}

// Canonical bit-reversed code of symbol t (tree.rs:102-177); false if the
// lengths form no code.
__device__ bool canonical(Scratch& S, uint32_t l, uint32_t& rev) {
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  // lane b: this wavefront's symbols of length b
  uint32_t rank = 0, mine = 0;
#pragma unroll 1
  for (uint32_t b = 1; b <= 11; ++b) {
    const uint64_t m = __ballot(l == b);
    if (l == b) rank = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    if (lane == b) mine = (uint32_t)__popcll(m);
  }
  if (lane < 16) S.count[wave][lane] = mine;
  __syncthreads();
  // lane b: the first code of length b, and the symbols of it in the
  // wavefronts before this one
  uint32_t count = 0, before = 0, first = 0;
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w) {
    const uint32_t c = S.count[w][lane & 15u];
    count += c;
    before += w < wave ? c : 0u;
  }
  uint32_t code = 0, prev = 0;
  bool ok = true;
#pragma unroll 1
  for (uint32_t b = 1; b <= 11; ++b) {
    const uint32_t c = lane_of(count, b);
    code = (code + prev) << 1;
    if (lane == b) first = code;
    // (past the longest length the reference does not look)
    if (c && code + c > (1u << b)) ok = false;
    prev = c;
  }
  const uint32_t at = (uint32_t)__shfl((int)(first + before), (int)l, 64) + rank;
  rev = l ? __builtin_bitreverse32(at) >> (32u - l) : 0u;
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
  const uint64_t used = __ballot(h != 0);
  if ((t & 63u) == 0) S.used[t >> 6] = used;
  __syncthreads();
  uint32_t n = 0, n_sym = 0, below = (uint32_t)__popcll(used & ((1ull << (t & 63u)) - 1ull));
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w) {
    const uint64_t m = S.used[w];
    if (w < t >> 6) below += (uint32_t)__popcll(m);
    n += (uint32_t)__popcll(m);
    if (m) n_sym = 64 * w + 64 - (uint32_t)__builtin_clzll(m);
  }
  uint8_t* const head = reinterpret_cast<uint8_t*>(S.head);
  bool ok = n != 0;
  uint32_t head_len = 0;
  if (ok && J.kind <= kTableIlv) {
    uint32_t rev;
    const uint32_t l = huffman_length(S, h, below, n, J.kind == kTableIlv && n_sym <= 16 ? 6u : 11u);
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
