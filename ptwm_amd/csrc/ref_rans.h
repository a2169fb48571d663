// ref_rans.h -- what bounds the bytes of a reference rANS segment
// (ref_encode.hip), apart so that it can be compiled and checked on the host.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ptwm {

// Bytes that state x sheds before the symbol of thresholds th: one if
// x >= freq << 20 and another if x >= freq << 28.  x is below 2^31 and both
// thresholds' low 16 bits are zero, so the upper half of x decides, below
// 2^15: th holds (freq << 4) - 1 and (min(freq, 8) << 12) - 1, and the
// signs of th - (x >> 16) are counted.
__host__ __device__ inline uint32_t shed(uint32_t x, uint32_t th) {
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  const u16x2 v = __builtin_bit_cast(u16x2, x);
  const u16x2 d = __builtin_bit_cast(u16x2, th) - v.yy;
  return (uint32_t)__builtin_popcount(__builtin_bit_cast(uint32_t, d) & 0x80008000u);
}

// The identity entry, of positions outside a segment and of the symbols of a
// refused table: {rcp, bias, cmpl | shift << 24, thresholds}.  It leaves a
// state below 2^31 as it is.
constexpr uint32_t kRansIdentityTh = 0x7FFF7FFFu;

// Scratch of a segment of n symbols: x_final, at most two bytes a symbol, and
// the two that an identity step after them sheds from a state of 2^31 or
// more.  The tables of the plane's own counts keep the state below that;
// entries that do not fit the symbols (bytes that change during the call) do
// not.
constexpr uint64_t ref_rans_scratch(uint64_t n) { return 4 + 2 * n + 2; }

}  // namespace ptwm
