// Index arithmetic that kernels and host share and that a host test goes through: plain C++, no HIP.
#pragma once
#include <stdint.h>

namespace pkh3 {

// rows of an operand-image buffer (pkh3_packed_bytes) that holds `rows` rows
constexpr int64_t padded_rows(int64_t rows) { return (rows + 255) / 256 * 256; }

// Whether the 16-row block that starts at `row` lies in such a buffer.  GEMM tiles of 256, 128 and 64 tokens end where it does or
// before; the last tile of 192 may reach up to 128 rows past it.
constexpr bool in_image_buffer(int row, int rows) { return row < padded_rows(rows); }

}  // namespace pkh3
