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

constexpr int kKvMaxHeads = 8;        // heads a workgroup of the K/V pass walks at most
constexpr int kOwnMaskKeys = 4096;    // keys whose mask a workgroup of the K/V pass can look through

// How the K/V pass splits the heads of a tile up: `groups` workgroups of each side walk `heads` heads each (the last one maybe fewer).
struct KvSplit {
  int heads, groups;
};
// More heads a workgroup share one read of the tables, as long as two or three workgroups of each side are left per CU.  15,342
// rows x 24 heads with rotation: 1 head 113 us, 2 91, 4 87, 8 85, 12 87; fp8 117, 90, 82, 76, 84.
// Three from where single heads make more workgroups than run at once (1, 2, 3 and 4 heads, us, 24 heads with rotation:
// 1,000 rows 9.8, 10.1, 9.2, 10.4; 1,500 13.7, 12.5, 12.2, 13.9; 3,000 24.8, 20.8, 20.1, 22.8, fp8 25.0, 22.0, 20.4, 22.9; without rotation
// 1,000 rows 7.1, 7.9, 7.8, 8.9; 1,500 9.8, 9.8, 9.6, 10.9; 3,000 18.6, 17.3, 17.0, 19.2).
constexpr KvSplit kv_split(int tiles, int batches, int heads, int cus) {
  const int64_t single = (int64_t)tiles * batches * heads;
  int64_t most = single * 2 / (5 * (int64_t)cus);
  if (most < 3 && single * 4 >= 9 * (int64_t)cus) most = 3;
  if (most > kKvMaxHeads) most = kKvMaxHeads;
  if (most > heads) most = heads;
  if (most < 1) most = 1;
  const int groups = (heads + (int)most - 1) / (int)most;
  const int n = (heads + groups - 1) / groups;   // equal shares
  return KvSplit{n, (heads + n - 1) / n};
}

// Whether the workgroups of the K/V pass look through the key mask themselves, each of them through all of it, or a launch of one
// workgroup an entry in front of the pass makes a list for them.  The launch costs about 1 us; the looks cost less while all
// workgroups run at once, and from there on they add up.  Launch / looks, us, with 2, 30 and 95 % of the keys valid: 24 heads x
// 512 keys (384 workgroups) 8.7 / 7.8, 9.1 / 8.2 and 10.2 / 9.3, 2 x 8 heads x 4,096 (768) 13.5 / 12.0, 14.8 / 14.1 and 21.1 / 19.8;
// 4 x 8 x 4,096 (1,536) 15.1 / 16.2, 19.8 / 21.3 and 32.1 / 34.5, 16 x 24 x 4,096 (6,144) 33.7 / 59.1, 116 / 133 and 313 / 321.  Of 492 such
// calls none of fewer than four workgroups a CU is faster with the launch.
constexpr bool kv_pass_reads_mask(int keys, int64_t workgroups, int cus) { return keys <= kOwnMaskKeys && workgroups < 4 * (int64_t)cus; }

}  // namespace pkh3
