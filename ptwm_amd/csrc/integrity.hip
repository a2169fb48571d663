// integrity.hip -- CRC-32/ISO-HDLC of device buffers (decoded planes).
//
// The reference checks each decoded plane against the CRC its record carries
// (container.rs:2154-2159: crc32fast::hash of the plane bytes, crc32fast
// 1.5.0 = reflected polynomial 0xEDB88320, init and final xor 0xFFFFFFFF).
//
// GPU formulation.  A zero-initialised CRC register is linear in the data,
// and advancing it over m zero bytes multiplies it by x^(8m) mod P.  So:
//   - each workgroup takes a range of a buffer; thread t owns the 16-byte
//     pieces t, t+256, ... (coalesced dwordx4 loads) and keeps one register
//     r, relative to the end of its latest piece: r' = r x^(8 * 4096) xor
//     crc0(piece), the advance by one 4 KiB tile as four byte-sliced
//     lookups and crc0 (the zero-init CRC of the 16 bytes, slicing-by-4,
//     Kounavis & Berry 2005) independent of r, so that the serial chain per
//     piece is one round of lookups;
//   - every thread's register is moved to the range end by one GF(2)
//     multiply with x^(8d) (d = its distance to the end) and the 256 values
//     are xor-reduced: the range's zero-init CRC, moved to the end of its
//     plane and XORed into the plane's accumulator;
//   - the launch's last workgroup hands the accumulators to the host
//     (crc_finish), which applies the init and final xor:
//     crc = ~(~0 * x^(8n) xor raw).
// The fused decodes add their blocks' CRCs to accumulators of the same kind.
#include "integrity.h"

#include "chain_ops.h"
#include "crc_device.h"

#include <algorithm>
#include <vector>

namespace ptwm {

namespace {

// One chain's tasks of a launch: a workgroup takes the range of rl plane
// bytes blockIdx.x, of the task whose ranges include it.  Up to kCrcInline
// tasks travel in the kernel arguments.
struct CrcTaskDev {
  uint64_t src, n;
  uint32_t first_range;  // range index of the task's first range
  uint32_t acc_ix;       // accumulator of its first plane
};
constexpr uint32_t kCrcInline = 8;
struct CrcTaskList {
  const CrcTaskDev* mem;  // m > kCrcInline
  uint64_t rl;
  uint32_t m, pad;
  CrcTaskDev t[kCrcInline];
};

std::vector<uint32_t> build_tables() {
  std::vector<uint32_t> tab(kCrcTabWords, 0);
  for (uint32_t i = 0; i < 256; ++i) {
    uint32_t c = i;
    for (int k = 0; k < 8; ++k) c = (c >> 1) ^ (kCrcPoly & (0u - (c & 1u)));
    tab[i] = c;
  }
  for (int k = 1; k < 4; ++k)
    for (uint32_t i = 0; i < 256; ++i) {
      const uint32_t prev = tab[256 * (k - 1) + i];
      tab[256 * k + i] = (prev >> 8) ^ tab[prev & 255u];
    }
  uint32_t* X = &tab[kCrcTabX];
  X[0] = kCrcOne >> 8;  // x^8
  for (int k = 1; k < 64; ++k) X[k] = gf2_mulmod(X[k - 1], X[k - 1]);
  const uint32_t adv = xpow8(kCrcTile, X);
  for (int k = 0; k < 4; ++k)
    for (uint32_t b = 0; b < 256; ++b) tab[kCrcTabS + 256 * k + b] = gf2_mulmod(b << (8 * k), adv);
  for (uint32_t t = 0; t < kCrcThreads; ++t) tab[kCrcTabK + t] = xpow8((uint64_t)kCrcPiece * (kCrcThreads - 1 - t), X);
  // accumulator element v of lane l: CRC bit l % 32 of row 8 (v / 4) +
  // 4 (l / 32) + v % 4, which ends 16 (31 - row) bytes before its half
  for (uint32_t l = 0; l < 64; ++l)
    for (uint32_t v = 0; v < 16; ++v) {
      const uint32_t row = 8 * (v / 4) + 4 * (l / 32) + v % 4;
      tab[kCrcTabRow + 256 * (v / 4) + 4 * l + v % 4] = gf2_mulmod(1u << (l % 32), xpow8(16ull * (31 - row), X));
    }
  const uint32_t z = xpow8(kCrcBlock, X);
  uint32_t zi = kCrcOne;
  for (uint32_t i = 0; i < 256; ++i, zi = gf2_mulmod(zi, z))
    for (uint32_t r = 0; r < 16; ++r) tab[kCrcTabW + 16 * i + r] = gf2_mulmod(zi, xpow8(1024 * (15 - r), X));
  uint32_t step = zi;  // Z^256
  for (uint32_t k = 0; k < 3; ++k) {
    uint32_t w = kCrcOne;
    for (uint32_t i = 0; i < 256; ++i, w = gf2_mulmod(w, step)) tab[kCrcTabZ + 256 * k + i] = w;
    step = w;
  }
  for (uint32_t k = 0; k < 5; ++k) {
    uint32_t w = kCrcOne;
    for (uint32_t i = 0; i < 256; ++i, w = gf2_mulmod(w, X[8 * k])) tab[kCrcTabQ + 256 * k + i] = w;
  }
  // the MFMA's constant operand: in lane 32 h + j's word, the bit of nibble i
  // that stands for data bit 4 i + q of half h's word holds bit j of what
  // that data bit contributes
  const uint32_t place[4] = {2u, 1u, 0u, 3u};  // crc_mma_const
  // bit b of a word that ends d bytes before the group's end
  auto bit_crc = [&](uint32_t b, uint64_t d) {
    const uint32_t w = 1u << b;
    const uint32_t c = tab[768 + (w & 255u)] ^ tab[512 + ((w >> 8) & 255u)] ^ tab[256 + ((w >> 16) & 255u)] ^ tab[w >> 24];
    return gf2_mulmod(c, xpow8(d, X));
  };
  for (uint32_t h = 0; h < 2; ++h)
    for (uint32_t s = 0; s < 16; ++s)
      for (uint32_t q = 0; q < 4; ++q)
        for (uint32_t i = 0; i < 8; ++i) {
          const uint32_t half = 512 * (1 - h), bit = 4 * i + place[q], lane = 32 * h;
          // byte planes: round s / 4, word s % 4
          const uint32_t cb = bit_crc(4 * i + q, 1024ull * (3 - s / 4) + half + 4 * (3 - s % 4));
          for (uint32_t j = 0; j < 32; ++j) tab[kCrcTabMmaB + s * 64 + lane + j] |= ((cb >> j) & 1u) << bit;
          if (s >= 8) continue;
          // nibble planes: round s / 2; nibble i of a word pair is byte i / 2 of word 2 (s % 2) + i % 2
          const uint32_t cn = bit_crc(8 * (i / 2) + q, 1024ull * (3 - s / 2) + half + 4 * (3 - 2 * (s % 2) - i % 2));
          for (uint32_t j = 0; j < 32; ++j) tab[kCrcTabMmaN + s * 64 + lane + j] |= ((cn >> j) & 1u) << bit;
        }
  return tab;
}

__device__ __forceinline__ uint32_t block_xor(uint32_t v, uint32_t* red) {
  for (int d = 32; d >= 1; d >>= 1) v ^= __shfl_xor(v, d, 64);
  if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return red[0] ^ red[1] ^ red[2] ^ red[3];
}

// Zero-init CRC of a range for every plane of its task, moved to the end of
// the plane and XORed into the plane's accumulator.  A range is a run of whole
// elements of one buffer; with kChain = passthrough the buffer is a plane
// itself, otherwise a restored tensor whose plane bytes are re-derived by the
// (bijective) forward chain.
template <uint32_t kChain>
__global__ void __launch_bounds__(256) crc_range_kernel(CrcTaskList L, CrcArgs args) {
  constexpr int kNp = kChain == kChainIeee16Split2 ? 2 : kChain == kChainIeee32Split4 ? 4 : 1;
  constexpr int kRatio = kNp;  // tensor bytes per plane byte for these chains
  __shared__ uint32_t tab[kCrcTabK];  // T0..T3, S0..S3
  __shared__ uint32_t red[4];
  __shared__ uint32_t flag;
  const uint32_t t = threadIdx.x;
  const uint32_t* const gtab = args.tab;
  for (uint32_t i = t; i < kCrcTabK; i += kCrcThreads) tab[i] = gtab[i];
  // the last task whose first range is not after this one
  CrcTaskDev J = L.t[0];
  if (L.m > kCrcInline) {
    uint32_t lo = 0, hi = L.m;
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) / 2;
      if (L.mem[mid].first_range <= blockIdx.x) lo = mid;
      else hi = mid;
    }
    J = L.mem[lo];
  } else {
#pragma unroll
    for (uint32_t k = 1; k < kCrcInline; ++k)
      if (k < L.m && L.t[k].first_range <= blockIdx.x) J = L.t[k];
  }
  struct {
    uint64_t src, n;
  } R;
  const uint64_t o = L.rl * (blockIdx.x - J.first_range);
  R.src = J.src + o * kRatio;
  R.n = std::min<uint64_t>(L.rl, J.n - o);
  __syncthreads();
  const uint32_t* T = tab;
  const uint32_t* S = tab + kCrcTabS;
  const uint64_t full = R.n / kCrcTile, tail = R.n % kCrcTile;
  const u32x4* p = reinterpret_cast<const u32x4*>(R.src) + (uint64_t)t * kRatio;
  uint32_t acc[kNp];
#pragma unroll
  for (int j = 0; j < kNp; ++j) acc[j] = 0;
  auto step = [&](uint64_t k) {
    u32x4 v[kRatio], pl[kNp];
#pragma unroll
    for (int h = 0; h < kRatio; ++h) v[h] = g_ld_nt16(reinterpret_cast<uint64_t>(p + k * kCrcThreads * kRatio + h));
    forward16<kChain>(v, pl);
#pragma unroll
    for (int j = 0; j < kNp; ++j) acc[j] = sliced(S, acc[j]) ^ crc_piece(T, 0u, pl[j]);
  };
  // four tiles per iteration, their loads issued before any lookup
  constexpr int kU = 4;
  uint64_t k = 0;
  for (; k + kU <= full; k += kU) {
    u32x4 v[kU][kRatio];
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int h = 0; h < kRatio; ++h)
        v[u][h] = g_ld_nt16(reinterpret_cast<uint64_t>(p + (k + u) * kCrcThreads * kRatio + h));
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      u32x4 pl[kNp];
      forward16<kChain>(v[u], pl);
#pragma unroll
      for (int j = 0; j < kNp; ++j) acc[j] = sliced(S, acc[j]) ^ crc_piece(T, 0u, pl[j]);
    }
  }
  for (; k < full; ++k) step(k);
  if (tail == 0) {
    if (full) {
      const uint32_t K = gtab[kCrcTabK + t];
#pragma unroll
      for (int j = 0; j < kNp; ++j) acc[j] = gf2_mulmod(acc[j], K);
    }
  } else {
    // the last, partial tile: thread t's piece may be whole, cut, or absent
    const uint64_t base = full * kCrcTile + (uint64_t)kCrcPiece * t;
    uint64_t end = full ? base - kCrcTile + kCrcPiece : 0;
    bool any = full != 0;
    if (base + kCrcPiece <= R.n) {
      step(full);
      end = base + kCrcPiece;
      any = true;
    } else if (base < R.n) {
      // the register advanced over the gap before this piece
      const uint32_t gap = full ? xpow8(kCrcTile - kCrcPiece, gtab + kCrcTabX) : 0u;
#pragma unroll
      for (int j = 0; j < kNp; ++j) {
        uint32_t c = gf2_mulmod(acc[j], gap);
        for (uint64_t i = base; i < R.n; ++i) c = T[(c ^ forward_byte<kChain>(R.src, i, j)) & 255u] ^ (c >> 8);
        acc[j] = c;
      }
      end = R.n;
      any = true;
    }
    if (any) {
      const uint32_t K = xpow8(R.n - end, gtab + kCrcTabX);
#pragma unroll
      for (int j = 0; j < kNp; ++j) acc[j] = gf2_mulmod(acc[j], K);
    }
  }
  uint32_t mine = 0;
#pragma unroll
  for (int j = 0; j < kNp; ++j) {
    const uint32_t v = block_xor(acc[j], red);
    if (t == (uint32_t)j) mine = v;
    __syncthreads();
  }
  if (t < (uint32_t)kNp) {
    uint64_t after = J.n - o - R.n;  // below 2^40 (crc_launch)
    for (uint32_t k = 0; after; ++k, after >>= 8)
      mine = gf2_mulmod_seq(mine, gtab[kCrcTabQ + 256 * k + (uint32_t)(after & 255u)]);
    __hip_atomic_fetch_xor(&args.acc[J.acc_ix + t], mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (args.n) crc_finish(args, &flag);
}

int chain_np(uint32_t chain) { return chain == kChainIeee16Split2 ? 2 : chain == kChainIeee32Split4 ? 4 : 1; }

hipError_t launch_crc_ranges(uint32_t chain, uint32_t cnt, const CrcTaskList& L, const CrcArgs& args, hipStream_t s) {
  const dim3 g(cnt), b(kCrcThreads);
  if (chain == kChainIeee16Split2) hipLaunchKernelGGL(crc_range_kernel<kChainIeee16Split2>, g, b, 0, s, L, args);
  if (chain == kChainIeee32Split4) hipLaunchKernelGGL(crc_range_kernel<kChainIeee32Split4>, g, b, 0, s, L, args);
  if (chain == kChainPassthrough) hipLaunchKernelGGL(crc_range_kernel<kChainPassthrough>, g, b, 0, s, L, args);
  return hipGetLastError();
}

const std::vector<uint32_t>& host_tables() {
  static const std::vector<uint32_t> t = build_tables();
  return t;
}

}  // namespace

bool crc_chain_supported(uint32_t chain) {
  return chain == kChainIeee16Split2 || chain == kChainIeee32Split4 || chain == kChainPassthrough;
}

static_assert(kNoAllocTabBytes >= kCrcTabWords * 4, "CRC tables fit the allocation-free scratch");
static_assert(kNoAllocAccBytes >= 4ull * (4ull * kNoAllocMaxTensors + kCrcAccHead), "CRC accumulators fit it");

int64_t crc_begin(DevCtx& ctx, uint32_t n, CrcArgs& args) {
  if (!ctx.crc_tab_ready) {
    const std::vector<uint32_t>& t = host_tables();
    PTWM_HIP_TRY(ctx.crc_tab.ensure(t.size() * 4));
    PTWM_HIP_TRY(hipMemcpyAsync(ctx.crc_tab.ptr, t.data(), t.size() * 4, hipMemcpyHostToDevice, ctx.stream));
    PTWM_HIP_TRY(hipStreamSynchronize(ctx.stream));
    ctx.crc_tab_ready = true;
  }
  const size_t need = 4ull * ((size_t)n + kCrcAccHead);
  const size_t before = ctx.crc_acc.cap;
  PTWM_HIP_TRY(ctx.crc_acc.ensure(need));
  // the accumulators are zero between calls: they are cleared when they are
  // new, and after a call that did not hand them over
  if (ctx.crc_acc.cap != before || ctx.crc_dirty)
    PTWM_HIP_TRY(hipMemsetAsync(ctx.crc_acc.ptr, 0, ctx.crc_acc.cap, ctx.stream));
  PTWM_HIP_TRY(ctx.h_crc.ensure(4ull * ((size_t)n + 1)));
  uint32_t* const out = static_cast<uint32_t*>(ctx.h_crc.ptr);
  out[n] = 0;
  ctx.crc_dirty = true;
  args.tab = static_cast<const uint32_t*>(ctx.crc_tab.ptr);
  args.done = static_cast<uint32_t*>(ctx.crc_acc.ptr);
  args.acc = args.done + kCrcAccHead;
  args.out = out;
  args.n = n;
  return kOk;
}

int64_t crc_take(DevCtx& ctx, const CrcArgs& args, std::vector<uint32_t>& raw) {
  if (args.out[args.n] != 1) return kInternal;
  raw.assign(args.out, args.out + args.n);
  ctx.crc_dirty = false;
  return kOk;
}

uint32_t crc_expected(uint32_t crc, uint64_t n, uint64_t unit) {
  const uint32_t* X = &host_tables()[kCrcTabX];
  const uint64_t padded = (n + unit - 1) / unit * unit;
  return gf2_mulmod(~crc, xpow8(padded - n, X)) ^ gf2_mulmod(0xFFFFFFFFu, xpow8(padded, X));
}

int64_t crc_launch(DevCtx& ctx, const std::vector<CrcTask>& tasks, CrcRun& run) {
  hipStream_t s = ctx.stream;
  // Range length (plane bytes): a multiple of the 4 KiB tile, sized so the
  // whole batch makes about 16 workgroups per CU.
  uint64_t total = 0;
  uint32_t n_acc = 0, parts = 0;
  for (const CrcTask& k : tasks) {
    if (!crc_chain_supported(k.chain)) return kInternal;
    if (k.n >> 40) return kInternal;             // more than the device holds
    if (k.n && (k.src & 15u)) return kInternal;  // callers pass 16-byte aligned buffers
    total += k.n * (uint64_t)chain_np(k.chain);
    n_acc += (uint32_t)chain_np(k.chain);
    parts += k.n != 0;
  }
  run.any = parts != 0;
  run.n = n_acc;
  if (!parts) return kOk;
  if (int64_t rc = crc_begin(ctx, n_acc, run.args); rc != kOk) return rc;
  const uint64_t cus = ctx.cu_count > 0 ? (uint64_t)ctx.cu_count : 256;
  uint64_t rl = (total / (cus * 16) + kCrcTile - 1) / kCrcTile * kCrcTile;
  rl = std::max<uint64_t>(rl, 16 * kCrcTile);
  rl = std::min<uint64_t>(rl, 1ull << 30);
  // one launch per chain, its tasks in the kernel arguments or in one upload
  const uint32_t chains[3] = {kChainIeee16Split2, kChainIeee32Split4, kChainPassthrough};
  std::vector<CrcTaskDev> dev[3];
  uint32_t cnt[3] = {0, 0, 0};
  uint32_t acc = 0;
  for (const CrcTask& k : tasks) {
    const int c = k.chain == kChainIeee16Split2 ? 0 : k.chain == kChainIeee32Split4 ? 1 : 2;
    if (k.n) {
      dev[c].push_back(CrcTaskDev{k.src, k.n, cnt[c], acc});
      cnt[c] += (uint32_t)((k.n + rl - 1) / rl);
    }
    acc += (uint32_t)chain_np(k.chain);
  }
  size_t up = 0;
  for (int c = 0; c < 3; ++c) up += dev[c].size() > kCrcInline ? dev[c].size() : 0;
  CrcTaskDev* d = nullptr;
  if (up) {
    PTWM_HIP_TRY(ctx.crc_args.ensure(up * sizeof(CrcTaskDev)));
    PTWM_HIP_TRY(ctx.h_crc_args.ensure(up * sizeof(CrcTaskDev)));
    CrcTaskDev* h = static_cast<CrcTaskDev*>(ctx.h_crc_args.ptr);
    d = static_cast<CrcTaskDev*>(ctx.crc_args.ptr);
    size_t o = 0;
    for (int c = 0; c < 3; ++c)
      if (dev[c].size() > kCrcInline) {
        std::copy(dev[c].begin(), dev[c].end(), h + o);
        o += dev[c].size();
      }
    PTWM_HIP_TRY(hipMemcpyAsync(d, h, up * sizeof(CrcTaskDev), hipMemcpyHostToDevice, s));
  }
  int final = 2;
  while (!cnt[final]) --final;
  for (int c = 0; c <= final; ++c) {
    if (!cnt[c]) continue;
    CrcTaskList L{};
    L.rl = rl;
    L.m = (uint32_t)dev[c].size();
    if (L.m > kCrcInline) {
      L.mem = d;
      d += L.m;
    } else {
      std::copy(dev[c].begin(), dev[c].end(), L.t);
    }
    CrcArgs a = run.args;
    if (c != final) a.n = 0;
    PTWM_HIP_TRY(launch_crc_ranges(chains[c], cnt[c], L, a, s));
  }
  return kOk;
}

int64_t crc_values(DevCtx& ctx, const CrcRun& run, std::vector<uint32_t>& raw) {
  raw.assign(run.n, 0);
  return run.any ? crc_take(ctx, run.args, raw) : kOk;
}

int64_t crc32_planes(DevCtx& ctx, const std::vector<CrcTask>& tasks, std::vector<uint32_t>& crcs) {
  CrcRun run;
  if (int64_t rc = crc_launch(ctx, tasks, run); rc != kOk) return rc;
  PTWM_HIP_TRY(hipStreamSynchronize(ctx.stream));
  if (int64_t rc = crc_values(ctx, run, crcs); rc != kOk) return rc;
  // crc = ~(raw xor ~0 x^(8 n)): crc_expected's inverse without padding
  size_t i = 0;
  for (const CrcTask& k : tasks) {
    const uint32_t init = crc_expected(0xFFFFFFFFu, k.n, 1);
    for (int j = 0; j < chain_np(k.chain); ++j, ++i) crcs[i] = ~(crcs[i] ^ init);
  }
  return kOk;
}

}  // namespace ptwm
