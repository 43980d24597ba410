// Index arithmetic and rules on sizes that a host test goes through besides the kernels and their launches: plain C++, no HIP.
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

// Tokens per workgroup of a launch of gemm_kernel (16 * 2 * TB).  Time of a CU's share of the launch, in units of 100 us for K = 3,072 with an
// adapter, from the workgroups it runs: one alone on the CU, and two (side by side for the smaller forms, one after the
// other for TB = 8).  Measured at 1,085, 15,342 and 48,360 tokens x 9,216 and 3,072 features: TB = 8 67 us alone, 79 - 84 us
// each in a long launch; TB = 6 53 and 104 us; TB = 4 40 us alone, 80 us for two; TB = 2 34 and 61 us.  What sets them: the smaller forms copy and
// read more for the same MFMAs (a chunk: 64, 48 and 40 KiB read and 32, 24 and 20 KiB copied for 256, 128 and 64 MFMAs) and have
// fewer of them between two barriers to cover a copy's way with, against how evenly their tiles fill the CUs.
// TB = 6 is for launches of one tile a CU, where 192 tokens fill them better than 256 or 128 (us, 256 / 192 / 128 tokens: 1,085 x 9,216
// 64.7 / 54.7 / 65.4, 3,000 x 3,072 63.9 / 52.9 / 64.8); in longer ones it is behind one of the others or the same (6,000 x 9,216 272 / 270 /
// 251, 6,000 x 3,072 131 / 104 / 104).  Where 64-token tiles come to two a CU, its start and end (12 us against 8.5) have to be made good over
// the chunks: from 64 of them on they are (1,305 x 6,144, K 96, 512, 1,024, 2,048 and 3,072: 192 tokens 13.1, 19.5, 26.0, 39.4 and 52.6, 64 tokens 10.0, 17.0,
// 24.0, 40.3 and 55.2; 1,540 x 5,120, K 2,048 39.7 and 39.5).
constexpr int gemm_token_blocks(int tokens, int n_tiles, int chunks, int cus) {
  constexpr struct { int tb; float one, two; } kForms[4] = {{8, 0.67f, 1.55f}, {6, 0.53f, 0.f}, {4, 0.40f, 0.80f}, {2, 0.34f, 0.61f}};
  int best = 8;
  float best_cost = 0.f;
  for (const auto& f : kForms) {
    const int tiles = (tokens + 32 * f.tb - 1) / (32 * f.tb) * n_tiles;
    const int per_cu = (tiles + cus - 1) / cus;
    if (f.tb == 6 && (per_cu > 1 || (chunks < 64 && (tokens + 63) / 64 * n_tiles <= 2 * cus))) continue;
    const float cost = (per_cu / 2) * f.two + (per_cu & 1) * f.one;
    if (f.tb == 8 || cost < best_cost) best = f.tb, best_cost = cost;
  }
  return best;
}

// The relay form of the attention kernel gives every workgroup a run of units, 128 queries each of one head after the other, and walks three
// units of a head in a round.  Units in front of the run of workgroup `rank`, in equal shares:
constexpr int relay_even_cut(int rank, int units, int wgs) { return rank * (units / wgs) + rank * (units % wgs) / wgs; }
constexpr int relay_rounds(int units) { return (units + 2) / 3; }
// ... and with a unit moved to the run before where that saves a round.  A run that crosses the end of a head has rounds of fewer than three
// units on both sides of it: eight of 256 workgroups took a round more than the others, which the call waits for, and a round is
// what the form gains.  24 heads, us, form in its place before / equal shares / now: 6,500 rows (51 units a head) x 512 keys 50.2 / 54.0 / 50.2,
// x 1,024 82.6 / 88.3 / 80.9; 14,830 (116) x 1,024 167 / 164.5 / 162.3; with rotation 3 x 24 x 2,000 (16) x 2,000 179 / 168 / 154.
// `fills`: also where the last round of the run before becomes one of three units.  With rotation, whose partial rounds are cheaper beside whole ones
// (waiting for the tables is the same), that lost what it saved: 14,830 x 1,088 189 -> 193, x 1,536 246.5 -> 250.
// (Runs of whole rounds throughout were worse, 49.5 -> 53.3 for 6,000 rows: a round of one unit takes 0.6 of one of three.)
constexpr int relay_cut(int rank, int units, int per_head, int wgs, bool fills) {
  const int at = relay_even_cut(rank, units, wgs);
  if (rank == 0 || rank >= wgs) return at;
  const int before = relay_even_cut(rank - 1, units, wgs), end = relay_even_cut(rank + 1, units, wgs);
  const int head = at / per_head * per_head, next = head + per_head;
  const bool crosses = before >= head && end > next && end <= next + per_head;   // one head's end, and the run before none
  const int most = relay_rounds((units + wgs - 1) / wgs), over = (at - before) % 3;
  if (!crosses || (next - at) % 3 != 1 || relay_rounds(next - at) + relay_rounds(end - next) <= most) return at;
  return over == 1 || (over == 2 && fills) ? at + 1 : at;                        // (the run before has no more rounds for it)
}
// Where the entries of a batch keep unequal keys, they are shared out by weight.  One of a batch entry takes as long as a third of a round,
// 3.9 us for its start and end and 2.1 to 2.2 for every key tile: two tiles' time besides the tiles.
constexpr int relay_weight(int valid_keys) { return (valid_keys + 63) / 64 + 2; }
// The unit of an entry of `units` units and weight `weight` that a workgroup begins with whose share begins into / wgs of a weight into it.  (One
// rounding of a number below 1 - 1 / 12,768, by which no unit past the end can come out.  Divisions of 64 bits in its place took about 1 us, 63 -> 64 of a call.)
constexpr int relay_unit(int into, int weight, int wgs, int units) { return (int)((float)into / (float)(weight * wgs) * (float)units); }

constexpr int kKvMaxHeads = 8;        // heads a workgroup of the K/V pass walks at most
constexpr int kOwnMaskKeys = 4096;    // keys whose mask a workgroup of the K/V pass can look through

// How the K/V pass splits the heads of a tile up: `groups` workgroups of each side walk `heads` heads each (the last one maybe fewer).
struct KvSplit {
  int heads, groups;
};
constexpr KvSplit kv_equal_split(int heads, int most) {
  const int groups = (heads + most - 1) / most, n = (heads + groups - 1) / groups;
  return KvSplit{n, (heads + n - 1) / n};
}
// More heads a workgroup share one read of the tables, as long as two or three workgroups of each side are left per CU.  15,342
// rows x 24 heads with rotation: 1 head 113 us, 2 91, 4 87, 8 85, 12 87; fp8 117, 90, 82, 76, 84.
// In between (2.5 to about 7 workgroups of single heads a side on a CU) it is the rounds that count: three workgroups of both sides
// run on a CU at once, and the fewest heads with which all of them do is best, if the heads in a row take no longer than the rounds
// they replace (a workgroup of n heads n + 1/2).  With rotation, whose tables are then read less often, already from 2.25 on and with
// up to five heads, else four; with a key mask three, as there are fewer tiles than the call says.
// This rule / three heads throughout / the rule above alone, us: 10 heads x 9,000 rows, fp8 27.3 / 30.9 / 27.3; 16 x 5,600, fp8 25.9 /
// 29.7 / 26.9; 24 x 3,000 20.1 / 20.1 / 24.8; 28 x 1,640 without rotation 12.8 / 14.7 / 13.8; 32 x 1,200 15.6 / 14.7 / 16.6; 4 heads x 16,384
// 19.6 / 21.6 / 25.9.  Of 504 such calls (4 to 48 heads) none that it sends another way is more than 0.5 % behind the rule above; of 137
// masked ones those with 10, 30, 60 and 95 % of the keys valid are 1, 2, 4 and 7 % ahead of it on average (at 10 and 30 % one in twelve
// 3 to 25 % behind).
constexpr KvSplit kv_split(int tiles, int batches, int heads, int cus, bool rotation, bool masked) {
  const int64_t single = (int64_t)tiles * batches * heads;
  int64_t most = single * 2 / (5 * (int64_t)cus);
  if (most > kKvMaxHeads) most = kKvMaxHeads;
  if (most > heads) most = heads;
  if (most < 1) most = 1;
  const KvSplit base = kv_equal_split(heads, (int)most);
  if (single * 4 < (rotation ? 9 : 10) * (int64_t)cus) return base;
  const int64_t side = (int64_t)tiles * batches, at_once = 3 * (int64_t)cus;
  const int64_t rounds = (2 * base.groups * side + at_once - 1) / at_once;
  for (int n = (int)most; n <= (masked ? 3 : rotation ? 5 : 4) && n <= heads; ++n) {
    const KvSplit s = kv_equal_split(heads, n);
    if (2 * s.groups * side <= at_once) return 2 * s.heads + 1 <= rounds * (2 * base.heads + 1) ? s : base;
  }
  return base;
}

// Whether the workgroups of the K/V pass look through the key mask themselves, each of them through all of it, or a launch of one
// workgroup an entry in front of the pass makes a list for them.  The launch costs about 1 us; the looks cost less while all
// workgroups run at once, and from there on they add up.  Launch / looks, us, with 2, 30 and 95 % of the keys valid: 24 heads x
// 512 keys (384 workgroups) 8.7 / 7.8, 9.1 / 8.2 and 10.2 / 9.3, 2 x 8 heads x 4,096 (768) 13.5 / 12.0, 14.8 / 14.1 and 21.1 / 19.8;
// 4 x 8 x 4,096 (1,536) 15.1 / 16.2, 19.8 / 21.3 and 32.1 / 34.5, 16 x 24 x 4,096 (6,144) 33.7 / 59.1, 116 / 133 and 313 / 321.  Of 492 such
// calls none of fewer than four workgroups a CU is faster with the launch.
constexpr bool kv_pass_reads_mask(int keys, int64_t workgroups, int cus) { return keys <= kOwnMaskKeys && workgroups < 4 * (int64_t)cus; }

}  // namespace pkh3
