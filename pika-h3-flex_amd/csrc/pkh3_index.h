// Index arithmetic that kernels and host share and that a host test goes through: plain C++, no HIP.
#pragma once
#include <stdint.h>

namespace pkh3 {

// rows of an operand-image buffer (pkh3_packed_bytes) that holds `rows` rows
constexpr int64_t padded_rows(int64_t rows) { return (rows + 255) / 256 * 256; }

// Whether the 16-row block that starts at `row` lies in such a buffer.  GEMM tiles of 256, 128 and 64 tokens end where it does or
// before; the last tile of 192 may reach up to 128 rows past it.
constexpr bool in_image_buffer(int row, int rows) { return row < padded_rows(rows); }

// Which of a list of words a thread of the K/V pass clears: every workgroup of its [batches][groups] has 256 of them, whether the list
// goes that far or not.  64 bits: 2^23 workgroups (2^24 keys of 16 entries of one head) have 2^31.
constexpr int64_t word_to_clear(unsigned batch, unsigned groups, unsigned group, unsigned thread) {
  return ((int64_t)batch * groups + group) * 256 + thread;
}

}  // namespace pkh3
