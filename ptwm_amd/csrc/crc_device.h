// crc_device.h -- CRC-32/ISO-HDLC building blocks shared by the CRC kernels
// (integrity.hip) and the fused decodes' CRCs of the planes they restore
// (huff_ilv.hip, rans_ilv.hip).  Reflected representation: bit 31 - i holds the x^i
// coefficient; a zero-initialised CRC register is linear in the data, and
// advancing it over m zero bytes multiplies it by x^(8m) mod P.
#pragma once

#include "ptwm_common.h"

namespace ptwm {

constexpr uint32_t kCrcPoly = 0xEDB88320u;  // reflected x^32 + x^26 + ... + 1; bit 31 = x^0
constexpr uint32_t kCrcOne = 0x80000000u;   // the polynomial 1
constexpr uint32_t kCrcPiece = 16, kCrcThreads = 256, kCrcTile = kCrcPiece * kCrcThreads;

// Bytes of a plane that one MFMA block covers (a codec block): the fused
// decodes' CRCs are linear combinations of whole blocks, the last one padded
// with zeros.
constexpr uint32_t kCrcBlock = 16384;

// Table layout in device memory (words):
//   kCrcTabT   T0..T3: one-byte table and its slicing-by-4 successors
//   kCrcTabS   S0..S3: byte-sliced advance over kCrcTile zero bytes
//   kCrcTabK   K[t] = x^(8 * 16 * (255 - t))
//   kCrcTabX   X[k] = x^(8 * 2^k)
//   kCrcTabRow [4][lane][4]: the weights of an MFMA accumulator's 16 elements
//   kCrcTabW   [256][16]: Z^i x^(8 * 1024 (15 - r)), Z = x^(8 * kCrcBlock)
//   kCrcTabZ   [3][256]: Z^(256 i), Z^(65536 i), Z^(2^24 i)
//   kCrcTabQ   [5][256]: x^(8 * 256^k i)
//   kCrcTabMmaB, kCrcTabMmaN: the MFMA's constant operand (crc_mma_word) for
//              planes of bytes, [4 rounds][4 words][lane], and for planes of
//              nibbles, [4 rounds][2 word pairs][lane]
constexpr uint32_t kCrcTabT = 0, kCrcTabS = 1024, kCrcTabK = 2048, kCrcTabX = 2304, kCrcTabRow = 2368,
                   kCrcTabW = 3392, kCrcTabZ = 7488, kCrcTabQ = 8256, kCrcTabMmaB = 9536, kCrcTabMmaN = 10560,
                   kCrcTabWords = 11072;
constexpr uint32_t kCrcMmaWordsB = 1024, kCrcMmaWordsN = 512;
constexpr uint32_t kCrcRowWords = 1024;  // words of kCrcTabRow
// LDS bytes of a launch with plane CRCs: the constant operand and the weights
constexpr uint32_t crc_lds_bytes(bool nib) { return 4u * ((nib ? kCrcMmaWordsN : kCrcMmaWordsB) + kCrcRowWords); }
static_assert(kCrcTabRow % 4 == 0 && kCrcTabMmaB % 4 == 0 && kCrcTabMmaN % 4 == 0, "16-byte loads");

// A launch's CRC arguments: the tables, the planes' accumulators (zero between
// calls), and for the last launch of a call (n > 0) what crc_finish needs.
struct CrcArgs {
  const uint32_t* tab;
  uint32_t* acc;
  uint32_t* done;  // workgroup counter, zero between launches
  uint32_t* out;   // host-coherent: n sums, then a 1
  uint32_t n;
  uint32_t pad;
};

// a * b mod P, reflected representation (bit 31 - i holds the x^i coefficient)
__host__ __device__ inline uint32_t gf2_mulmod(uint32_t a, uint32_t b) {
  uint32_t p = 0;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    p ^= b & (0u - ((a >> (31 - i)) & 1u));
    b = (b >> 1) ^ (kCrcPoly & (0u - (b & 1u)));
  }
  return p;
}

// The same, computed as a short loop: unrolled whole, the compiler keeps
// all 32 shifted multiples of b in registers at once, which in a kernel
// that needs its registers elsewhere costs occupancy.
__device__ __forceinline__ uint32_t gf2_mulmod_seq(uint32_t a, uint32_t b) {
  uint32_t p = 0;
#pragma unroll 4
  for (int i = 0; i < 32; ++i) {
    p ^= b & (0u - (a >> 31));
    a <<= 1;
    b = (b >> 1) ^ (kCrcPoly & (0u - (b & 1u)));
  }
  return p;
}

// x^(8 n) mod P from the squares table X (X[k] = x^(8 * 2^k))
__host__ __device__ inline uint32_t xpow8(uint64_t n, const uint32_t* X) {
  uint32_t r = kCrcOne;
  for (int k = 0; n; ++k, n >>= 1)
    if (n & 1u) r = gf2_mulmod(r, X[k]);
  return r;
}

__device__ __forceinline__ uint32_t sliced(const uint32_t* L, uint32_t c) {
  return L[c & 255u] ^ L[256 + ((c >> 8) & 255u)] ^ L[512 + ((c >> 16) & 255u)] ^ L[768 + (c >> 24)];
}

// one word through the one-byte tables T0..T3 (T3 takes the first byte)
__device__ __forceinline__ uint32_t crc_word(const uint32_t* T, uint32_t c, uint32_t w) {
  c ^= w;
  return T[768 + (c & 255u)] ^ T[512 + ((c >> 8) & 255u)] ^ T[256 + ((c >> 16) & 255u)] ^ T[c >> 24];
}

__device__ __forceinline__ uint32_t crc_piece(const uint32_t* T, uint32_t c, u32x4 v) {
  c = crc_word(T, c, v.x);
  c = crc_word(T, c, v.y);
  c = crc_word(T, c, v.z);
  return crc_word(T, c, v.w);
}

// ---- the fused decodes' CRC on the matrix cores ----
// A plane's CRC is a GF(2)-linear map of its bits: a 0/1 matrix product whose
// sums are taken mod 2.  One v_mfma_f32_32x32x64 with FP4 operands takes a
// 32-bit word of plane data from every lane (row lane % 32, the lane's half
// of the wavefront picking one of two 32-wide slices of K) against a constant
// operand whose column j holds bit j of each data bit's CRC contribution, and
// adds the 32 rows' CRC bits, as counts, to the accumulator.  The counts
// start at 2^23, where an f32's last mantissa bit is the integer's parity, and
// never pass 2^23 + 1024, so they are exact.
//
// Lane 32 h + i holds piece i of half h of each 1 KiB round: its distance to
// the round's end is folded into the constant operand for h and the word, and
// into the accumulator elements' weights (kCrcTabRow) for i.  The constant
// operand covers the rounds of one group (4 rounds), a bit per element in LDS
// (4 KiB; a nibble plane's words carry two data words: 2 KiB), opened to FP4
// where it is used: every KiB more takes wavefronts off the CU, which the
// decode's chains of table lookups need more than the CRC needs fewer groups.
// At a group's end the accumulator becomes one CRC word (crc_mma_close).
//
// Against byte-sliced table lookups (20 scattered LDS reads, 20 address
// shifts and 20 XORs per 16 bytes and lane) this takes 4 LDS reads without
// bank conflicts, 20 VALU instructions and 4 MFMAs, and 4 reads and 20
// instructions more that all planes share.  Measured on whole calls: four
// bf16 layers (1.74 GB) 878 -> 750 us; the nibble and rans_ilv tensors, whose
// CRCs were passes of their own before, e4m3 8192 x 8192 186 -> 87 us and
// fp32 4096 x 4096 153 -> 96 us.  The call waits for the device once (before:
// again for each of the range and combine kernels and their uploads): one
// norm weight 98 -> 43 us.
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x16 crc_mma_open() {
  f32x16 c;
#pragma unroll
  for (int i = 0; i < 16; ++i) c[i] = 8388608.0f;
  return c;
}

// Add the word t against the constant operand's word b.  Bit 4 i + q of t is
// nibble i of data register q: bits 0, 1 and 2 of each nibble masked in place
// (the FP4 values 0.5, 1 and 2), bit 3 moved to 2; the constant operand holds
// the reciprocals, so its bits for q = 0, 1, 2, 3 are nibble bits 2, 1, 0, 3.
__device__ __forceinline__ i32x8 crc_mma_operand(u32x4 v) {  // (FP4: the first four registers)
  return __builtin_bit_cast(i32x8, __builtin_shufflevector(v, v, 0, 1, 2, 3, -1, -1, -1, -1));
}
__device__ __forceinline__ i32x8 crc_mma_const(uint32_t b) {
  return crc_mma_operand(u32x4_make(b & 0x44444444u, b & 0x22222222u, b & 0x11111111u, (b >> 3) & 0x11111111u));
}
__device__ __forceinline__ void crc_mma_word(f32x16& c, uint32_t t, i32x8 b) {
  const i32x8 a =
      crc_mma_operand(u32x4_make(t & 0x11111111u, t & 0x22222222u, t & 0x44444444u, (t >> 1) & 0x44444444u));
  // cbsz = blgp = 4: FP4; zero scale operands: the unscaled instruction
  c = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 4, 4, 0, 0, 0, 0);
}

// XOR over the wavefront's 64 lanes, in lane 63 (all lanes active): the rows
// of 16 by row shifts, then broadcasts of rows 0, 2 (to 1, 3) and of row 1
// (to 2, 3).
__device__ __forceinline__ uint32_t wave_xor63(uint32_t v) {
  v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true);
  v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, true);
  v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, true);
  v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, true);
  v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);
  v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);
  return v;
}

// One wavefront's CRC state for the block it decodes.  Plane p's CRC of the
// bytes up to the end of round r (and from the last such lane's on) is left
// in lane 4 r + p; crc_block_add weights all of them at once.
struct CrcLane {
  uint32_t row;      // LDS address of the accumulator weights
  uint32_t mma;      // LDS address of the constant operand
  uint32_t val;
  uint32_t last;     // blocks after block 0 of the tensor
  uint32_t sum;      // lane p: plane p's CRC of the wavefront's blocks so far
};

// The planes' CRCs of a group (uniform): the parity of an accumulator's
// element v selects its weight.
template <uint32_t NP>
__device__ __forceinline__ void crc_mma_close(const f32x16 (&c)[NP], uint32_t row, uint32_t lane, uint32_t (&x)[NP]) {
#pragma unroll
  for (uint32_t p = 0; p < NP; ++p) x[p] = 0;
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    const u32x4 w = *(const __attribute__((address_space(3))) u32x4*)(uintptr_t)(row + 1024u * k + 16u * lane);
#pragma unroll
    for (uint32_t p = 0; p < NP; ++p)
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) x[p] ^= (0u - (__float_as_uint(c[p][4 * k + i]) & 1u)) & w[i];
  }
#pragma unroll
  for (uint32_t p = 0; p < NP; ++p) x[p] = (uint32_t)__builtin_amdgcn_readlane((int)wave_xor63(x[p]), 63);
}

// Add the block's plane CRCs, moved to the end of the plane, to the
// wavefront's sums: block bi has e = last - bi blocks after it, so its bytes
// are weighted by Z^e.
__device__ __forceinline__ void crc_block_add(CrcLane& cl, uint32_t bi, const uint32_t* tab, uint32_t lane) {
  const uint32_t e = cl.last - bi;
  uint32_t a = gf2_mulmod_seq(cl.val, tab[kCrcTabW + 16u * (e & 255u) + (lane >> 2)]);
  for (uint32_t k = 0, r = e >> 8; r; ++k, r >>= 8) a = gf2_mulmod_seq(a, tab[kCrcTabZ + 256u * k + (r & 255u)]);
#pragma unroll
  for (int d = 4; d < 64; d <<= 1) a ^= __shfl_xor(a, d, 64);
  cl.sum ^= a;
}

// At the end of a tensor (or of the launch): every wavefront adds its sums to
// the workgroup's in LDS (crc_sum_up), and after a barrier four threads XOR
// those into the accumulators (crc_sum_out).  One atomic per workgroup, plane
// and tensor: with one per block (8192 for a 64 MiB e4m3 tensor, all to one
// line) that tensor's kernel took 82 us against 56.
__device__ __forceinline__ void crc_sum_up(CrcLane& cl, uint32_t* sums, uint32_t lane) {
  if (lane < 4 && cl.sum) __hip_atomic_fetch_xor(&sums[lane], cl.sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  cl.sum = 0;
}
__device__ __forceinline__ void crc_sum_out(uint32_t* sums, uint32_t* acc, uint32_t acc_ix) {
  const uint32_t t = threadIdx.x;
  if (t >= 4) return;
  const uint32_t v = sums[t];
  sums[t] = 0;
  if (v) __hip_atomic_fetch_xor(&acc[acc_ix + t], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The end of a kernel whose workgroups XOR into acc[0..n): the last one to
// get here moves the sums to host-coherent memory (out[0..n), then out[n] = 1)
// and leaves the accumulators and the counter zero for the next launch.  Every
// thread of every workgroup of the launch calls it once, after its last
// addition.  flag: a word of LDS.
__device__ __forceinline__ void crc_finish(const CrcArgs& a, volatile uint32_t* flag) {
  // this thread's additions have been performed (vector memory operations
  // count until they are)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t wgs = gridDim.x * gridDim.y;
    *flag = wgs == 1 || __hip_atomic_fetch_add(a.done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == wgs - 1;
  }
  __syncthreads();
  if (!*flag) return;
  for (uint32_t i = threadIdx.x; i < a.n; i += blockDim.x)
    __hip_atomic_store(&a.out[i], __hip_atomic_exchange(&a.acc[i], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (threadIdx.x == 0) {
    __hip_atomic_store(a.done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&a.out[a.n], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

}  // namespace ptwm
