// huffman_host.h -- Huffman code lengths on the host.
#pragma once

#include <cstdint>

namespace ptwm {

constexpr int kHufMaxBits = 11;  // MAX_TABLE_LOG (entropy/huffman/tree.rs:5)

// Code lengths from a histogram (tree.rs:19-85 + enforce_max_code_length
// :212-242 at max_len, the reference encoder's 11 by default).  Returns false
// when every count is zero.
bool huf_lengths_from_freqs(const uint32_t freqs[256], uint8_t lengths[256], int max_len = kHufMaxBits);

}  // namespace ptwm
