// code_tables.h -- entropy code tables built on the device (code_tables.hip).
#pragma once

#include "ptwm_common.h"

namespace ptwm {

// What a table is for.
enum TableKind : uint32_t {
  kTableHuffman = 0,  // the reference's Huffman code (11-bit limit)
  kTableIlv = 1,      // huff_ilv's: a 6-bit limit when every symbol is below 16
  kTableRans = 2,     // the reference's rANS frequencies and encoder symbols
  kTableRansIlv = 3,  // rans_ilv's: the same frequencies, f | cum << 16 per symbol
};

// Table j of a launch: the histogram is the sum of `rows` (0 to 4) rows of 256 counts
// from row `row0` on.  Its codes go to codes[256 j ..] (kTableHuffman /
// kTableIlv: length << 16 | bit-reversed code; kTableRansIlv: f | cum << 16)
// or rans[256 j ..] (kTableRans).
struct TableJob {
  uint32_t kind, row0, rows, pad;
};

// What the host needs of it, written to host-coherent memory.
struct alignas(16) TableInfo {
  uint32_t ok;        // the table exists (0: no symbols, or no valid code)
  uint32_t n_sym;     // last symbol with a nonzero count, plus one
  uint32_t head_len;  // bytes of `head`
  uint32_t pad;
  uint64_t bits[4];   // Huffman: code bits of each row; kTableRansIlv: [0], rans_ilv_least
  uint8_t head[528];  // the payload's table header (weights, or max_sym and frequencies)
};

hipError_t launch_code_tables(const TableJob* jobs, uint32_t n, const uint32_t* hist, uint32_t* codes, uint4* rans,
                              TableInfo* info, hipStream_t stream);

}  // namespace ptwm
