// ref_encode.hip -- GPU encoder for the reference's Huffman and rANS plane
// payloads, byte-identical to the reference encoder.
//
// Payload framing: codecs/huffman.rs:37-87 and codecs/rans.rs:38-94
// ([00] empty, [00]+raw when not beneficial, [01][orig_len u32][blob]);
// blobs: entropy/huffman/compress.rs:9-103 (weights header, jump table,
// four backward bitstreams over split_four segments) and
// entropy/rans/compress.rs:128-260 (frequency header, jump table, four
// streams [x_final u32][renorm bytes in decoder order]).
//
// One call encodes a batch of jobs (each one payload: a whole plane or one
// chunk of a chunked plane):
//   1. histogram per job (ref_hist_kernel);
//   2. code tables per job (code_tables.hip: the reference tree, canonical
//      codes and weights header; rANS: normalize_freqs and the EncSymbol
//      reciprocal parameters of rans/compress.rs:35-122);
//   3. Huffman: bits per segment from the segment's histogram and the code
//      lengths (the histograms are taken per split_four segment); rANS:
//      each segment encoded into scratch (ref_rans_kernel; a segment's
//      state chain is serial by construction);
//   4. host: payload sizes, coded-or-raw decisions, output layout;
//   5. Huffman segments packed in parallel: every symbol's bit offset is a
//      prefix sum of code lengths, so each segment is cut into slices of
//      kSliceSyms symbols, the bits of every slice summed
//      (ref_huf_slice_bits_kernel) and scanned per segment
//      (ref_huf_slice_scan_kernel), and every slice packed from its offset
//      by its own workgroup (ref_huf_pack_kernel); then headers, streams
//      and raw fallbacks placed by one gather launch of 64 KiB pieces
//      (ref_copy_kernel).
#include "ref_encode.h"

#include <algorithm>
#include <cstring>

#include "code_tables.h"
#include "ref_rans.h"

namespace ptwm {

namespace {

constexpr uint32_t kRansL = 1u << 23;

__device__ __forceinline__ uint8_t gbyte(uint64_t a) {
  return *(const __attribute__((address_space(1))) uint8_t*)(uintptr_t)a;
}

// a word store at any address
__device__ __forceinline__ void g_st_u32_any(uint64_t a, uint32_t v) {
  typedef uint32_t __attribute__((aligned(1))) u32_any;
  *(__attribute__((address_space(1))) u32_any*)(uintptr_t)a = v;
}

// atomic OR into global memory (not a flat atomic: see g_ld)
__device__ __forceinline__ void or_global(uint32_t* p, uint32_t v) {
  __hip_atomic_fetch_or((__attribute__((address_space(1))) uint32_t*)(uintptr_t)p, v, __ATOMIC_RELAXED,
                        __HIP_MEMORY_SCOPE_AGENT);
}

// 256-bin histogram per job (blockIdx.y); any source alignment.
__global__ void __launch_bounds__(256) ref_hist_kernel(const RefJobDev* __restrict__ jobs, uint32_t* __restrict__ hist) {
  __shared__ uint32_t h[4][256];
  const RefJobDev J = jobs[blockIdx.y];
  const uint32_t t = threadIdx.x, wave = t >> 6;
  for (uint32_t i = t; i < 1024; i += 256) (&h[0][0])[i] = 0;
  __syncthreads();
  const uint64_t head = J.n == 0 ? 0 : std::min<uint64_t>(J.n, (16 - (J.src & 15)) & 15);
  const uint64_t nvec = (J.n - head) / 16;
  const uint64_t stride = (uint64_t)gridDim.x * 256u;
  const u32x4* v = reinterpret_cast<const u32x4*>(J.src + head);
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + t; i < nvec; i += stride) {
    const u32x4 x = g_ld_nt16(reinterpret_cast<uint64_t>(v + i));
    const uint32_t xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int b = 0; b < 4; ++b) atomicAdd(&h[wave][(xs[k] >> (8 * b)) & 0xFF], 1u);
  }
  if (blockIdx.x == 0) {
    for (uint64_t i = t; i < head; i += 256) atomicAdd(&h[wave][gbyte(J.src + i)], 1u);
    for (uint64_t i = head + nvec * 16 + t; i < J.n; i += 256) atomicAdd(&h[wave][gbyte(J.src + i)], 1u);
  }
  __syncthreads();
  const uint32_t s = h[0][t] + h[1][t] + h[2][t] + h[3][t];
  if (s) atomicAdd(&hist[256u * blockIdx.y + t], s);
}

// Huffman: total code bits of each slice.  The slice's bytes are read as the
// aligned words that hold them, one word per thread per step.
__global__ void __launch_bounds__(256) ref_huf_slice_bits_kernel(const RefSegDev* __restrict__ segs,
                                                                 const RefSliceDev* __restrict__ slices,
                                                                 const uint32_t* __restrict__ codes,
                                                                 unsigned long long* __restrict__ slice_bits) {
  __shared__ uint8_t len[256];
  __shared__ unsigned long long part[4];
  const RefSliceDev L = slices[blockIdx.x];
  const RefSegDev S = segs[L.seg];
  const uint32_t t = threadIdx.x;
  len[t] = (uint8_t)(codes[256u * S.table + t] >> 16);
  __syncthreads();
  const uint64_t b0 = S.src + L.sym0, b1 = b0 + L.n, a0 = b0 & ~3ull;
  unsigned long long bits = 0;
  for (uint64_t a = a0 + 4ull * t; a < b1; a += 1024) {
    const uint32_t w = g_ld<uint32_t>(a);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
      if (a + k >= b0 && a + k < b1) bits += len[(w >> (8 * k)) & 0xFFu];
  }
  for (int d = 32; d >= 1; d >>= 1) bits += __shfl_down(bits, d, 64);
  if ((t & 63u) == 0) part[t >> 6] = bits;
  __syncthreads();
  if (t == 0) slice_bits[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// Exclusive scan of each segment's slice bits (workgroup g: the slices
// [first[g], first[g + 1])), in place: each slice's starting bit.
__global__ void __launch_bounds__(256) ref_huf_slice_scan_kernel(const uint32_t* __restrict__ first,
                                                                 unsigned long long* __restrict__ slice_bits) {
  __shared__ unsigned long long wsum[4];
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  const uint32_t s0 = first[blockIdx.x], s1 = first[blockIdx.x + 1];
  unsigned long long carry = 0;
  for (uint32_t b = s0; b < s1; b += 256) {
    const uint32_t i = b + t;
    const unsigned long long v = i < s1 ? slice_bits[i] : 0ull;
    unsigned long long incl = v;
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
      const unsigned long long o = __shfl_up(incl, d, 64);
      if (lane >= d) incl += o;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    unsigned long long before = 0, tot = 0;
    for (uint32_t w = 0; w < 4; ++w) {
      if (w < wave) before += wsum[w];
      tot += wsum[w];
    }
    if (i < s1) slice_bits[i] = carry + before + incl - v;
    carry += tot;
    __syncthreads();
  }
}

// Huffman: pack one segment's codes (bit-reversed canonical codes,
// LSB-first, bitstream.rs:22-50) straight into their final byte order.  The
// logical stream P (bit k = bit k % 8 of byte k / 8) is stored reversed
// (S[m-1-i] = P[i]); in the segment's word-aligned scratch area of W words
// whose last m bytes are S, logical word w is the byte-swapped word W-1-w.
// One workgroup per slice (slice_off: the slice's first bit).  Each pass
// covers 256 x kPackPerThread symbols: every thread reads its symbols as
// the aligned words that hold them, a workgroup scan gives each thread its
// bit offset, the pass's words are assembled in LDS (OR), and written out:
// the pass's first and last word with a global OR (they may be shared with
// the neighbouring pass or slice; the area starts zeroed), the others with
// plain stores.
constexpr uint32_t kPackPerThread = 8;
constexpr uint32_t kPackWords = (256u * kPackPerThread * 11u + 31u) / 32u + 2u;
__global__ void __launch_bounds__(256) ref_huf_pack_kernel(const RefSegDev* __restrict__ segs,
                                                           const RefSliceDev* __restrict__ slices,
                                                           const unsigned long long* __restrict__ slice_off,
                                                           const uint32_t* __restrict__ codes,
                                                           uint32_t* __restrict__ scratch) {
  __shared__ uint32_t code[256];
  __shared__ uint32_t wave_sum[4];
  __shared__ uint32_t asm_w[kPackWords];
  const RefSliceDev L = slices[blockIdx.x];
  const RefSegDev S = segs[L.seg];
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  code[t] = codes[256u * S.table + t];
  unsigned long long base = slice_off[blockIdx.x];
  uint32_t* area = scratch + S.scratch_word;
  const uint64_t W = S.words;
  const uint64_t src = S.src + L.sym0, end = src + L.n;
  __syncthreads();
  for (uint64_t pass = 0; pass < L.n; pass += 256ull * kPackPerThread) {
    for (uint32_t k = t; k < kPackWords; k += 256) asm_w[k] = 0;
    // this thread's symbols: bytes [a, a + 8) of the slice, from the three
    // aligned words that hold them (a word is read only if it starts
    // before the slice's end, so it holds one of the slice's bytes)
    const uint64_t a = src + pass + (uint64_t)t * kPackPerThread;
    const uint64_t aw = a & ~3ull;
    const uint32_t sh = (uint32_t)(a & 3u);
    uint32_t w[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) w[k] = aw + 4u * k < end ? g_ld<uint32_t>(aw + 4u * k) : 0u;
    const uint32_t lo = __builtin_amdgcn_alignbyte(w[1], w[0], sh), hi = __builtin_amdgcn_alignbyte(w[2], w[1], sh);
    uint32_t sym_code[kPackPerThread];
    uint32_t bits = 0;
#pragma unroll
    for (uint32_t k = 0; k < kPackPerThread; ++k) {
      const uint32_t b = ((k < 4 ? lo : hi) >> (8 * (k & 3))) & 0xFFu;
      sym_code[k] = a + k < end ? code[b] : 0u;
      bits += sym_code[k] >> 16;
    }
    // exclusive prefix of bits over the workgroup
    uint32_t incl = bits;
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
      const uint32_t o = __shfl_up(incl, d, 64);
      if (lane >= d) incl += o;
    }
    if (lane == 63) wave_sum[wave] = incl;
    __syncthreads();
    uint32_t before = 0, pass_bits = 0;
    for (uint32_t v = 0; v < 4; ++v) {
      if (v < wave) before += wave_sum[v];
      pass_bits += wave_sum[v];
    }
    // LDS word j holds the pass's logical word (base >> 5) + j
    const uint32_t b0 = (uint32_t)(base & 31u);
    uint32_t off = b0 + before + (incl - bits);
    uint32_t j = off >> 5, fill = off & 31u;
    uint64_t acc = 0;
#pragma unroll
    for (uint32_t k = 0; k < kPackPerThread; ++k) {
      acc |= (uint64_t)(sym_code[k] & 0xFFFFu) << fill;
      fill += sym_code[k] >> 16;
      if (fill >= 32) {
        atomicOr(&asm_w[j], (uint32_t)acc);
        acc >>= 32;
        fill -= 32;
        ++j;
      }
    }
    if (fill) atomicOr(&asm_w[j], (uint32_t)acc);
    __syncthreads();
    const uint32_t nw = (b0 + pass_bits + 31u) >> 5;
    const uint64_t w0 = base >> 5;
    for (uint32_t k = t; k < nw; k += 256) {
      uint32_t* dst = area + (W - 1 - (w0 + k));
      const uint32_t v = __builtin_bswap32(asm_w[k]);
      if (k == 0 || k + 1 == nw) or_global(dst, v);
      else g_st<uint32_t>(reinterpret_cast<uint64_t>(dst), v);
    }
    base += pass_bits;
    __syncthreads();
  }
}

// rANS: each segment encoded backward (encode_stream_into,
// rans/compress.rs:140-185) into its scratch area: [x_final u32 LE][renorm
// bytes in emission order]; seg_len = 4 + renorm bytes.  Table entries per
// symbol: {rcp, bias, cmpl | shift << 24, the two thresholds} (the
// thresholds: see shed).
//
// The state chain is serial by the format, and a wavefront issues one
// instruction per 5.2 cycles whether they depend on each other or not, so
// the kernel's time is a segment's symbols times the instructions of a step
// in the wave that holds the states.  That wave (wave 0, one lane per
// segment) is left with the state alone, eight instructions and one table
// entry read from a fixed place; the two other waves work beside it on the
// batches (kRansEncBatch symbols, aligned, last first) before and after:
// - wave 2 loads the symbols, two batches ahead, and lays their entries in
//   LDS in the order of the steps (identity entries for positions outside
//   the segment, which so need no test);
// - wave 1 takes the states of the batch before and stores the bytes that
//   they shed (four lanes per segment, each with a quarter of the steps).
// A workgroup has sixteen segments: with their entries, three batches of
// 8 KiB, LDS allows three workgroups per CU, and the entry reads and the
// stores, each lane's at its own address, stay far below the chain's time.
// A 16 MiB plane in 256 KiB chunks, 65536 steps, takes 2.0 ms: 70 cycles a
// step, 52 of them the state's (3.3 ms, 122 cycles, with one wave doing all).
constexpr uint32_t kRansEncSegs = 16;                    // segments per workgroup
constexpr uint32_t kRansEncJobs = kRansEncSegs / 4 + 1;  // job tables a workgroup can span
constexpr uint32_t kRansEncBatch = 32;                   // steps
constexpr uint32_t kRansEncThreads = 192;

__global__ void __launch_bounds__(kRansEncThreads) ref_rans_kernel(const RefSegDev* __restrict__ segs, uint32_t n_segs,
                                                                   const u32x4* __restrict__ tables,
                                                                   uint8_t* __restrict__ scratch,
                                                                   unsigned long long* __restrict__ seg_len) {
  constexpr uint32_t N = kRansEncSegs, B = kRansEncBatch;
  __shared__ u32x4 tab[kRansEncJobs][257];  // + the identity entry
  __shared__ u32x4 ent[3][B][N];            // a batch's entries, step by step
  __shared__ u32x4 state[2][B / 4][N];      // the states before its steps
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t n_here = min(N, n_segs - blockIdx.x * N);
  const uint32_t g = lane & (N - 1);  // this lane's segment (in waves 1 and 2, with three others)
  const RefSegDev S = segs[blockIdx.x * N + min(g, n_here - 1)];
  // A job's four segments are consecutive, so the workgroup's segments form
  // runs of one job each (at most kRansEncJobs): run r's table goes to tab[r].
  const uint32_t prev_job = (uint32_t)__shfl((int)S.table, (int)(g ? g - 1 : 0), 64);
  const uint64_t starts = __ballot(lane < N && (g == 0 || prev_job != S.table));
  const uint32_t slot = (uint32_t)__popcll(starts & ((2ull << g) - 1)) - 1;
  uint64_t rest = starts;
  for (uint32_t r = 0; rest; ++r) {
    const uint32_t at = (uint32_t)__builtin_ctzll(rest);
    rest &= rest - 1;
    const uint32_t jr = (uint32_t)__builtin_amdgcn_readlane((int)S.table, at);
    for (uint32_t i = threadIdx.x; i < 256; i += kRansEncThreads) tab[r][i] = tables[256ull * jr + i];
    if (threadIdx.x == 0) tab[r][256] = u32x4_make(0u, 0u, 0u, kRansIdentityTh);
  }
  // Batch b of the segment: the symbols of the aligned block top - b B.
  const uint64_t n = g < n_here ? S.n : 0;
  const uint64_t first = S.src, end = S.src + n;  // symbols [first, end)
  const uint64_t top = n ? (end - 1) & ~(uint64_t)(B - 1) : 0;
  const uint64_t count = n ? (top - (first & ~(uint64_t)(B - 1))) / B + 1 : 0;
  uint64_t batches = count;
  for (uint32_t d = 1; d < N; d <<= 1) batches = max(batches, (uint64_t)__shfl_xor((unsigned long long)batches, d, 64));
  batches = (uint64_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)batches) |
            (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(batches >> 32)) << 32;
  const uint64_t out = reinterpret_cast<uint64_t>(scratch + S.scratch_byte);
  __syncthreads();  // the tables

  // Wave 2, lane (c, g): symbol words c and c + 4 of the batch's eight.  A
  // word is read if it holds a symbol of the segment: an aligned word that
  // holds one byte in bounds is in bounds.
  const uint32_t c = lane / N;
  auto word_at = [&](uint64_t b, uint32_t k) { return top - b * B + 4 * k; };
  auto load = [&](uint64_t b, uint32_t k) -> uint32_t {
    const uint64_t a = word_at(b, k);
    return b < count && a < end && a + 4 > first ? g_ld<uint32_t>(a) : 0u;
  };
  auto lay = [&](uint64_t b, uint32_t buf, uint32_t k, uint32_t w) {
    const uint64_t a = word_at(b, k);
    const u32x4* const T = tab[slot];
    uint32_t sym[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) sym[i] = (w >> (8 * i)) & 0xFFu;
    if (!(b < count && a >= first && a + 4 <= end))
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i)
        if (!(b < count && a + i >= first && a + i < end)) sym[i] = 256;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) ent[buf][B - 1 - (4 * k + i)][g] = T[sym[i]];
  };
  uint32_t w0 = 0, w1 = 0, v0 = 0, v1 = 0;  // words of the next batch, and of the one after it
  if (wave == 2) {
    w0 = load(0, c), w1 = load(0, c + 4);
    v0 = load(1, c), v1 = load(1, c + 4);
  }
  uint32_t x = kRansL;     // wave 0
  uint32_t last = 0;       // wave 1: the last four bytes of the stream
  uint64_t pos = out + 4;  //         and its end
  uint32_t buf = 0;        // b mod 3
  // Pass b: batch b laid, batch b - 1 coded, batch b - 2 stored.
  for (uint64_t b = 0; b < batches + 2; ++b) {
    const uint32_t buf1 = buf == 0 ? 2 : buf - 1, buf2 = buf == 2 ? 0 : buf + 1;  // of b - 1, b - 2
    if (wave == 2) {
      const uint32_t n0 = load(b + 2, c), n1 = load(b + 2, c + 4);
      if (b < batches) {
        lay(b, buf, c, w0);
        lay(b, buf, c + 4, w1);
      }
      w0 = v0, w1 = v1, v0 = n0, v1 = n1;
    } else if (wave == 0 && b >= 1 && b <= batches) {
      // all four lanes of a segment do the same: with 16 active lanes a step
      // takes 63 cycles, with 64 of them 52
      const u32x4(*E)[N] = ent[buf1];
      u32x4(*X)[N] = state[(b - 1) & 1];
      u32x4 e[8], f[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) e[i] = E[i][g];
#pragma unroll
      for (uint32_t q = 0; q < B / 8; ++q) {
        // the next eight entries are read in the first four steps, and
        // waited for once: a wait at each step's entry costs as much as an
        // instruction
        asm("" : "+v"(e[0]), "+v"(e[1]), "+v"(e[2]), "+v"(e[3]), "+v"(e[4]), "+v"(e[5]), "+v"(e[6]), "+v"(e[7]));
        if (q + 1 < B / 8)
#pragma unroll
          for (int i = 0; i < 8; ++i) f[i] = E[8 * (q + 1) + i][g];
        uint32_t s[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {  // one step (rans/compress.rs:150-167)
          s[i] = x;
          const uint32_t xs = __builtin_amdgcn_alignbyte(0u, x, shed(x, e[i].w));
          x = xs + e[i].y + __umul24(__umulhi(xs, e[i].x) >> (e[i].z >> 24), e[i].z);
        }
        X[2 * q][g] = u32x4_make(s[0], s[1], s[2], s[3]);
        X[2 * q + 1][g] = u32x4_make(s[4], s[5], s[6], s[7]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);              // the pk_sub
          if (i < 4) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // in the slot after it
          __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = f[i];
      }
    } else if (wave == 1 && b >= 2) {
      // Lane (c, g): steps 8 c .. 8 c + 7.  What `last` is before each
      // lane's steps comes from the lanes below; then two steps shed at most
      // four bytes, those that `last` holds after them, and the word stores
      // at each two steps' end write right bytes only, also where they
      // overlap a lower lane's.
      const u32x4(*E)[N] = ent[buf2];
      const u32x4(*X)[N] = state[b & 1];
      const u32x4 xa = X[2 * c][g], xb = X[2 * c + 1][g];
      const uint32_t s[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
      uint32_t k[8], mine = 0, m = 0;  // bytes shed in the step, by the lane; its last four
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) k[i] = shed(s[i], E[8 * c + i][g].w);
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) {
        m = __builtin_amdgcn_alignbyte(s[i], m, k[i]);
        mine += k[i];
      }
      uint32_t before = 0, total = 0, l = last;
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        const uint32_t nj = (uint32_t)__shfl((int)mine, (int)(N * j + g), 64);
        const uint32_t mj = (uint32_t)__shfl((int)m, (int)(N * j + g), 64);
        if (j == c) before = total, last = l;
        l = mj | (nj < 4 ? l >> (8 * nj) : 0u);
        total += nj;
      }
      uint64_t at = pos + before;
      pos += total;
#pragma unroll
      for (uint32_t i = 0; i < 8; i += 2) {
        last = __builtin_amdgcn_alignbyte(s[i], last, k[i]);
        last = __builtin_amdgcn_alignbyte(s[i + 1], last, k[i + 1]);
        at += k[i] + k[i + 1];
        if (n) g_st_u32_any(at - 4, last);
      }
      last = l;
    }
    buf = buf == 2 ? 0 : buf + 1;
    __syncthreads();
  }
  if (wave == 1 && lane < n_here) seg_len[blockIdx.x * N + g] = pos - out;
  // the stream's first stores reach x_final's bytes too: after them
  if (wave == 0) state[0][0][g].x = x;
  __syncthreads();
  if (wave == 1 && lane < n_here) g_st<uint32_t>(out, state[0][0][g].x);
}

// Byte copies of a batch of ranges: bytes [0, rev_from) forward, bytes
// [rev_from, n) taken from the end of the source backward (the rANS renorm
// bytes, emitted in the reverse of decoder order).
// The forward part is copied in whole destination words: each is the
// source's bytes at any alignment, taken from the aligned source words that
// hold them (a source word is read only when it holds one of the bytes).
__global__ void __launch_bounds__(256) ref_copy_kernel(const RefCopyOp* __restrict__ ops) {
  const RefCopyOp op = ops[blockIdx.x];
  const uint32_t t = threadIdx.x;
  const uint64_t fwd = op.rev_from < op.n ? op.rev_from : op.n;
  const uint64_t head = std::min<uint64_t>(fwd, (4u - (op.dst & 3u)) & 3u);
  const uint64_t nw = (fwd - head) / 4;
  for (uint64_t i = t; i < head; i += 256) g_st<uint8_t>(op.dst + i, gbyte(op.src + i));
  for (uint64_t w = t; w < nw; w += 256) {
    const uint64_t sa = op.src + head + 4 * w, a = sa & ~3ull;
    const uint32_t sh = (uint32_t)(sa & 3u);
    const uint32_t w0 = g_ld<uint32_t>(a), w1 = sh ? g_ld<uint32_t>(a + 4) : 0u;
    g_st<uint32_t>(op.dst + head + 4 * w, __builtin_amdgcn_alignbyte(w1, w0, sh));
  }
  for (uint64_t i = head + 4 * nw + t; i < fwd; i += 256) g_st<uint8_t>(op.dst + i, gbyte(op.src + i));
  for (uint64_t i = fwd + t; i < op.n; i += 256) g_st<uint8_t>(op.dst + i, gbyte(op.src + op.n - 1 - (i - fwd)));
}

void split_four(uint64_t len, uint64_t start[4], uint64_t n[4]) {
  const uint64_t q = len / 4, r = len % 4;
  uint64_t off = 0;
  for (int i = 0; i < 4; ++i) {
    start[i] = off;
    n[i] = q + (i < (int)r ? 1 : 0);
    off += n[i];
  }
}

inline void put32(std::vector<uint8_t>& v, uint32_t x) {
  for (int i = 0; i < 4; ++i) v.push_back((uint8_t)(x >> (8 * i)));
}

inline uint64_t align_up(uint64_t v, uint64_t a) { return (v + a - 1) / a * a; }

}  // namespace

int64_t RefEncoder::plan(DevCtx& ctx, const std::vector<RefJob>& jobs, std::vector<uint64_t>& payload_len) {
  hipStream_t s = ctx.stream;
  jobs_ = jobs;
  const uint32_t nj = (uint32_t)jobs.size();
  payload_len.assign(nj, 0);
  info_.assign(nj, JobInfo{});
  segs_.clear();
  if (nj == 0) return kOk;
  // ---- 1. histograms, one per split_four segment (stream_frame.rs:11-62),
  // 2. the jobs' tables, 3. the rANS segments, with one wait at the end ----
  std::vector<RefJobDev> jd;
  std::vector<TableJob> tj(nj, TableJob{kTableHuffman, 0, 0, 0});
  std::vector<RefSegDev> rsegs;  // the rANS segments, and their indexes in segs_
  std::vector<uint32_t> ridx;
  uint64_t max_n = 0, scratch_words = 0, rans_scratch = 0;
  for (uint32_t j = 0; j < nj; ++j) {
    if (jobs[j].codec != kCodecHuffman && jobs[j].codec != kCodecRans) return kUnsupported;
    JobInfo& I = info_[j];
    I.raw = true;
    const uint64_t n = jobs[j].n;
    // (past 32 bits no payload is coded, and the table build adds counts in 32
    // bits: its merge may not end once its sums wrap several times)
    if (n == 0 || n > 0xFFFFFFFFull) continue;
    const bool rans = jobs[j].codec == kCodecRans;
    tj[j] = TableJob{rans ? kTableRans : kTableHuffman, (uint32_t)jd.size(), 4, 0};
    uint64_t st[4], sn[4];
    split_four(n, st, sn);
    I.raw = false;
    I.seg0 = (uint32_t)segs_.size();
    for (int i = 0; i < 4; ++i) {
      jd.push_back(RefJobDev{jobs[j].src + st[i], sn[i]});
      RefSegDev g{};
      g.src = jobs[j].src + st[i];
      g.n = sn[i];
      g.table = j;
      if (rans) {
        g.scratch_byte = rans_scratch;
        rans_scratch = align_up(rans_scratch + ref_rans_scratch(sn[i]), 16);
        ridx.push_back((uint32_t)segs_.size());
        rsegs.push_back(g);
      }
      segs_.push_back(g);
    }
    max_n = std::max(max_n, sn[0]);
  }
  const uint32_t ns = (uint32_t)segs_.size(), nr = (uint32_t)rsegs.size();
  seg_len_.assign(ns, 0);
  if (ns) {
    const size_t b_jd = ns * sizeof(RefJobDev), b_tj = nj * sizeof(TableJob), b_rs = nr * sizeof(RefSegDev);
    PTWM_HIP_TRY(ctx.ref_jobs.ensure(b_jd + b_tj + b_rs));
    PTWM_HIP_TRY(ctx.h_ref.ensure(b_jd + b_tj + b_rs));
    PTWM_HIP_TRY(ctx.ref_hist.ensure((size_t)ns * 256 * sizeof(uint32_t)));
    PTWM_HIP_TRY(ctx.ref_codes.ensure((size_t)nj * 256 * sizeof(uint32_t)));
    PTWM_HIP_TRY(ctx.h_tables.ensure(nj * sizeof(TableInfo) + nr * sizeof(unsigned long long)));
    if (nr) {
      PTWM_HIP_TRY(ctx.ref_rans_tab.ensure((size_t)nj * 256 * sizeof(uint4)));
      PTWM_HIP_TRY(ctx.ref_rans_scratch.ensure(rans_scratch));
    }
    uint8_t* const h = static_cast<uint8_t*>(ctx.h_ref.ptr);
    std::memcpy(h, jd.data(), b_jd);
    std::memcpy(h + b_jd, tj.data(), b_tj);
    if (nr) std::memcpy(h + b_jd + b_tj, rsegs.data(), b_rs);
    uint8_t* const d = static_cast<uint8_t*>(ctx.ref_jobs.ptr);
    TableInfo* const info = static_cast<TableInfo*>(ctx.h_tables.ptr);
    unsigned long long* const rlen = reinterpret_cast<unsigned long long*>(info + nj);
    uint32_t* const hist = static_cast<uint32_t*>(ctx.ref_hist.ptr);
    uint4* const rtab = static_cast<uint4*>(ctx.ref_rans_tab.ptr);
    PTWM_HIP_TRY(hipMemcpyAsync(d, h, b_jd + b_tj + b_rs, hipMemcpyHostToDevice, s));
    PTWM_HIP_TRY(hipMemsetAsync(hist, 0, (size_t)ns * 256 * sizeof(uint32_t), s));
    uint64_t hb = (max_n / 16 + 255) / 256;
    hb = std::max<uint64_t>(1, std::min<uint64_t>(hb, 256));
    for (uint32_t j0 = 0; j0 < ns; j0 += 65535) {
      const uint32_t cnt = std::min<uint32_t>(65535, ns - j0);
      hipLaunchKernelGGL(ref_hist_kernel, dim3((uint32_t)hb, cnt), dim3(256), 0, s,
                         reinterpret_cast<const RefJobDev*>(d) + j0, hist + 256ull * j0);
      PTWM_HIP_TRY(hipGetLastError());
    }
    PTWM_HIP_TRY(launch_code_tables(reinterpret_cast<const TableJob*>(d + b_jd), nj, hist,
                                    static_cast<uint32_t*>(ctx.ref_codes.ptr), rtab, info, s));
    if (nr) {
      hipLaunchKernelGGL(ref_rans_kernel, dim3((nr + kRansEncSegs - 1) / kRansEncSegs), dim3(kRansEncThreads), 0, s,
                         reinterpret_cast<const RefSegDev*>(d + b_jd + b_tj), nr, reinterpret_cast<const u32x4*>(rtab),
                         static_cast<uint8_t*>(ctx.ref_rans_scratch.ptr), rlen);
      PTWM_HIP_TRY(hipGetLastError());
    }
    PTWM_HIP_TRY(hipStreamSynchronize(s));
    for (uint32_t j = 0; j < nj; ++j) {
      JobInfo& I = info_[j];
      if (I.raw) continue;
      const TableInfo& T = info[j];
      if (!T.ok) {
        I.raw = true;
        continue;
      }
      I.header.assign(T.head, T.head + T.head_len);
      if (jobs[j].codec != kCodecHuffman) continue;
      for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t g = I.seg0 + i;
        seg_len_[g] = (T.bits[i] + 7) / 8;
        segs_[g].words = (T.bits[i] + 31) / 32;
        segs_[g].scratch_word = scratch_words;
        scratch_words += segs_[g].words + 1;
      }
    }
    for (uint32_t k = 0; k < nr; ++k) {
      const uint32_t g = ridx[k];
      if (info_[segs_[g].table].raw) continue;
      if (rlen[k] < 4) return kInternal;  // every rANS stream holds at least x_final
      seg_len_[g] = rlen[k];
    }
  }
  pack_words_ = scratch_words;
  // ---- 4. sizes and coded-or-raw (codecs/huffman.rs:50-87, codecs/rans.rs:50-94) ----
  for (uint32_t j = 0; j < nj; ++j) {
    JobInfo& I = info_[j];
    const uint64_t n = jobs[j].n;
    if (n == 0) {
      payload_len[j] = 1;  // [00]
      continue;
    }
    if (!I.raw) {
      uint64_t blob = I.header.size() + 16;
      for (int i = 0; i < 4; ++i) blob += seg_len_[I.seg0 + i];
      bool coded = blob < n;  // NotBeneficial when blob >= len (compress.rs:72-75)
      for (int i = 0; i < 4; ++i) coded = coded && seg_len_[I.seg0 + i] <= 0xFFFFFFFFull;
      // length_prefix::accepted (codecs/length_prefix.rs:15-56), rANS only
      if (coded && jobs[j].codec == kCodecRans) coded = n <= (1ull << 30) || n <= blob * 64;
      if (coded) {
        I.blob = blob;
        payload_len[j] = 5 + blob;
        continue;
      }
      I.raw = true;
    }
    payload_len[j] = 1 + n;  // [00] + plane
  }
  return kOk;
}

int64_t RefEncoder::write(DevCtx& ctx, const std::vector<uint64_t>& dst,
                          const std::vector<std::pair<uint64_t, std::vector<uint8_t>>>& literal,
                          const std::vector<RefCopyOp>& copies) {
  hipStream_t s = ctx.stream;
  const uint32_t nj = (uint32_t)jobs_.size();
  if (dst.size() != nj) return kInternal;
  // headers: [tag][orig_len][table header][jump table] per coded job, [00] per raw job
  std::vector<uint8_t> hdr;
  std::vector<uint64_t> hdr_off(nj + 1, 0);
  for (uint32_t j = 0; j < nj; ++j) {
    const JobInfo& I = info_[j];
    hdr_off[j] = hdr.size();
    if (I.raw) {
      hdr.push_back(0);
      continue;
    }
    hdr.push_back(1);
    put32(hdr, (uint32_t)jobs_[j].n);
    hdr.insert(hdr.end(), I.header.begin(), I.header.end());
    for (int i = 0; i < 4; ++i) put32(hdr, (uint32_t)seg_len_[I.seg0 + i]);
  }
  hdr_off[nj] = hdr.size();
  std::vector<uint64_t> lit_off;
  for (const auto& l : literal) {
    lit_off.push_back(hdr.size());
    hdr.insert(hdr.end(), l.second.begin(), l.second.end());
  }
  PTWM_HIP_TRY(ctx.ref_hdr.ensure(hdr.size() + 16));
  if (!hdr.empty()) PTWM_HIP_TRY(hipMemcpyAsync(ctx.ref_hdr.ptr, hdr.data(), hdr.size(), hipMemcpyHostToDevice, s));
  // Huffman segments packed into zeroed word scratch
  if (pack_words_) {
    PTWM_HIP_TRY(ctx.ref_pack.ensure(pack_words_ * 4));
    PTWM_HIP_TRY(hipMemsetAsync(ctx.ref_pack.ptr, 0, pack_words_ * 4, s));
    std::vector<RefSegDev> hs;
    std::vector<RefSliceDev> sl;
    std::vector<uint32_t> first;
    for (const RefSegDev& g : segs_) {
      if (jobs_[g.table].codec != kCodecHuffman || info_[g.table].raw || !g.n) continue;
      first.push_back((uint32_t)sl.size());
      for (uint64_t a = 0; a < g.n; a += kSliceSyms)
        sl.push_back(RefSliceDev{a, std::min<uint64_t>(kSliceSyms, g.n - a), (uint32_t)hs.size(), {0, 0, 0}});
      hs.push_back(g);
    }
    first.push_back((uint32_t)sl.size());
    if (!hs.empty()) {
      if (sl.size() > 0x7FFFFFFFull) return kInternal;
      const size_t b_seg = hs.size() * sizeof(RefSegDev), b_sl = sl.size() * sizeof(RefSliceDev);
      PTWM_HIP_TRY(ctx.ref_segs.ensure(b_seg + b_sl + first.size() * 4));
      PTWM_HIP_TRY(ctx.ref_seglen.ensure(sl.size() * sizeof(unsigned long long)));
      uint8_t* d = static_cast<uint8_t*>(ctx.ref_segs.ptr);
      PTWM_HIP_TRY(hipMemcpyAsync(d, hs.data(), b_seg, hipMemcpyHostToDevice, s));
      PTWM_HIP_TRY(hipMemcpyAsync(d + b_seg, sl.data(), b_sl, hipMemcpyHostToDevice, s));
      PTWM_HIP_TRY(hipMemcpyAsync(d + b_seg + b_sl, first.data(), first.size() * 4, hipMemcpyHostToDevice, s));
      const RefSegDev* d_seg = reinterpret_cast<const RefSegDev*>(d);
      const RefSliceDev* d_sl = reinterpret_cast<const RefSliceDev*>(d + b_seg);
      const uint32_t* d_first = reinterpret_cast<const uint32_t*>(d + b_seg + b_sl);
      unsigned long long* d_bits = static_cast<unsigned long long*>(ctx.ref_seglen.ptr);
      const uint32_t* d_codes = static_cast<const uint32_t*>(ctx.ref_codes.ptr);
      hipLaunchKernelGGL(ref_huf_slice_bits_kernel, dim3((uint32_t)sl.size()), dim3(256), 0, s, d_seg, d_sl, d_codes,
                         d_bits);
      hipLaunchKernelGGL(ref_huf_slice_scan_kernel, dim3((uint32_t)hs.size()), dim3(256), 0, s, d_first, d_bits);
      hipLaunchKernelGGL(ref_huf_pack_kernel, dim3((uint32_t)sl.size()), dim3(256), 0, s, d_seg, d_sl,
                         static_cast<const unsigned long long*>(d_bits), d_codes,
                         static_cast<uint32_t*>(ctx.ref_pack.ptr));
      PTWM_HIP_TRY(hipGetLastError());
    }
  }
  // gather: headers, streams, raw planes
  std::vector<RefCopyOp> ops;
  const uint64_t hdr_dev = reinterpret_cast<uint64_t>(ctx.ref_hdr.ptr);
  for (size_t k = 0; k < literal.size(); ++k)
    if (!literal[k].second.empty())
      ops.push_back(RefCopyOp{hdr_dev + lit_off[k], literal[k].first, literal[k].second.size(), ~0ull});
  // forward copies in pieces of at most kPiece bytes, one workgroup each
  constexpr uint64_t kPiece = 64ull << 10;
  const auto forward = [&](uint64_t src, uint64_t dst_addr, uint64_t n) {
    for (uint64_t o = 0; o < n; o += kPiece)
      ops.push_back(RefCopyOp{src + o, dst_addr + o, std::min<uint64_t>(kPiece, n - o), ~0ull});
  };
  for (const RefCopyOp& c : copies) forward(c.src, c.dst, c.n);
  for (uint32_t j = 0; j < nj; ++j) {
    const JobInfo& I = info_[j];
    const uint64_t hl = hdr_off[j + 1] - hdr_off[j];
    ops.push_back(RefCopyOp{hdr_dev + hdr_off[j], dst[j], hl, ~0ull});
    if (I.raw) {
      forward(jobs_[j].src, dst[j] + 1, jobs_[j].n);
      continue;
    }
    uint64_t o = dst[j] + hl;
    for (int i = 0; i < 4; ++i) {
      const RefSegDev& g = segs_[I.seg0 + i];
      const uint64_t m = seg_len_[I.seg0 + i];
      if (m) {
        if (jobs_[j].codec == kCodecHuffman) {
          // the stream is the last m bytes of the segment's word area
          const uint64_t area = reinterpret_cast<uint64_t>(ctx.ref_pack.ptr) + 4 * g.scratch_word;
          forward(area + 4 * g.words - m, o, m);
        } else {
          const uint64_t area = reinterpret_cast<uint64_t>(ctx.ref_rans_scratch.ptr) + g.scratch_byte;
          ops.push_back(RefCopyOp{area, o, m, 4});
        }
      }
      o += m;
    }
  }
  if (!ops.empty()) {
    PTWM_HIP_TRY(ctx.ref_ops.ensure(ops.size() * sizeof(RefCopyOp)));
    PTWM_HIP_TRY(hipMemcpyAsync(ctx.ref_ops.ptr, ops.data(), ops.size() * sizeof(RefCopyOp), hipMemcpyHostToDevice, s));
    for (size_t k0 = 0; k0 < ops.size(); k0 += 65535) {
      const uint32_t cnt = (uint32_t)std::min<size_t>(65535, ops.size() - k0);
      hipLaunchKernelGGL(ref_copy_kernel, dim3(cnt), dim3(256), 0, s,
                         static_cast<const RefCopyOp*>(ctx.ref_ops.ptr) + k0);
      PTWM_HIP_TRY(hipGetLastError());
    }
  }
  PTWM_HIP_TRY(hipStreamSynchronize(s));
  return kOk;
}

}  // namespace ptwm
