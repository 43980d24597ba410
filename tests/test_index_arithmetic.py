"""Index arithmetic and rules on sizes where they can go wrong, in a host build of the header the kernels share: no GPU needed."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pika-h3-flex_amd", "csrc")


def _run(tmp_path, body):
    """Builds and runs a program around ``body``, with the signed overflow and the bounds of constants checked."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "host.cc", tmp_path / "host"
    src.write_text('#include "pkh3_index.h"\n#include <stdio.h>\nusing namespace pkh3;\n'
                   '#define CHECK(x, ...) do { if (!(x)) { printf(__VA_ARGS__); return 1; } } while (0)\n'
                   "int main() {\n" + body + "\n  return 0;\n}\n")
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=undefined", "-fno-sanitize-recover", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout + done.stderr


def test_down_projected_images_stay_in_their_buffer(tmp_path):
    """Tiles of 64, 128, 192 and 256 tokens, two waves each, 16-row blocks: every block with a token is written, none past the buffer."""
    _run(tmp_path, """
  for (int rows = 1; rows <= 3 * 768; ++rows)
    for (int blocks = 2; blocks <= 8; blocks += 2)
      for (int first = 0; first < rows; first += 16 * blocks) {   // a wave; waves without a token write nothing
        for (int row = first; row < first + 16 * blocks; row += 16) {
          if (row < rows) CHECK(in_image_buffer(row, rows), "%d rows: block at %d is left out", rows, row);
          if (blocks != 6 || in_image_buffer(row, rows))
            CHECK(row + 16 <= padded_rows(rows), "%d rows, %d a tile: block at %d", rows, 32 * blocks, row);
        }
      }""")


def test_words_cleared_by_the_kv_pass_are_those_of_the_list(tmp_path):
    """Grids from the smallest that clears the longest list (6,208 words) to those of the largest calls that are accepted: the first
    workgroups clear every word once, no index is negative and none comes twice."""
    _run(tmp_path, """
  struct { unsigned batches, groups; } grids[] = {{1, 34}, {17, 2}, {65535, 130}, {16, 524288}, {17, 524288}, {65535, 524288}};
  for (auto g : grids) {
    const int64_t all = (int64_t)g.batches * g.groups;
    for (int64_t word = 0; word < 6208; ++word) {
      const int64_t wg = word / 256;
      CHECK(word_to_clear(wg / g.groups, g.groups, wg % g.groups, word % 256) == word, "word %lld", (long long)word);
    }
    for (int64_t wg = all > 70000 ? all - 70000 : 25; wg < all; ++wg)
      CHECK(word_to_clear(wg / g.groups, g.groups, wg % g.groups, 0) == wg * 256, "workgroup %lld of %lld", (long long)wg, (long long)all);
    for (int64_t wg = 25; wg < all; wg += all / 1000 + 1)
      CHECK(word_to_clear(wg / g.groups, g.groups, wg % g.groups, 0) >= 6208, "workgroup %lld of %lld", (long long)wg, (long long)all);
  }""")


def test_who_reads_the_key_mask(tmp_path):
    """The K/V pass where its workgroups run at once (measured on 256 CUs), a launch in front of it for more of them or more keys."""
    _run(tmp_path, """
  struct { int keys, heads, entries; bool pass; } calls[] = {
      {512, 24, 1, true}, {777, 8, 3, true}, {512, 24, 4, true}, {4096, 8, 2, true}, {4096, 1, 7, true},
      {4097, 1, 1, false}, {4096, 1, 8, false}, {4096, 8, 4, false}, {1000, 4, 16, false}, {4096, 24, 16, false}, {300, 24, 64, false}};
  for (auto c : calls) {
    const int tiles = (c.keys + 63) / 64;
    const KvSplit split = kv_split(tiles, c.entries, c.heads, 256, false, true);
    CHECK(split.groups * split.heads >= c.heads && (split.groups - 1) * split.heads < c.heads, "%d heads", c.heads);
    CHECK(kv_pass_reads_mask(c.keys, (int64_t)2 * split.groups * tiles * c.entries, 256) == c.pass, "%d keys, %d x %d", c.keys, c.entries, c.heads);
  }""")


def test_heads_a_workgroup_of_the_kv_pass(tmp_path):
    """Calls that three heads a workgroup were slower for than the fewest with which all workgroups run at once, or than as many as fill
    the CUs (measured on 256 CUs); every head is somebody's at any size."""
    _run(tmp_path, """
  struct { int tiles, heads; bool rotation; int want; bool masked; } calls[] = {
      {141, 10, true, 2}, {167, 10, true, 5}, {88, 16, true, 4}, {72, 10, false, 2}, {45, 16, false, 2}, {26, 28, false, 2}, {144, 5, false, 1},
      {50, 12, false, 1}, {47, 24, true, 3}, {47, 24, false, 3}, {16, 24, true, 1}, {240, 24, true, 8}, {8, 24, false, 1}, {256, 4, true, 4}, {256, 4, true, 1, true}, {47, 24, true, 3, true}};
  for (auto c : calls) {
    const KvSplit s = kv_split(c.tiles, 1, c.heads, 256, c.rotation, c.masked);
    CHECK(s.heads == c.want, "%d tiles, %d heads: %d a workgroup", c.tiles, c.heads, s.heads);
  }
  for (int tiles = 1; tiles < 300; tiles += 7)
    for (int heads = 1; heads <= 70; ++heads)
      for (int rotation = 0; rotation < 2; ++rotation) {
        const KvSplit s = kv_split(tiles, 1 + heads % 3, heads, 256, rotation, tiles % 2);
        CHECK(s.heads >= 1 && s.heads <= kKvMaxHeads && s.groups * s.heads >= heads && (s.groups - 1) * s.heads < heads, "%d tiles, %d heads", tiles, heads);
      }""")


def test_tokens_a_workgroup_of_the_projections(tmp_path):
    """On 256 CUs: 192 tokens for launches of one such tile a CU, of few chunks only where 64-token tiles come to more than two."""
    _run(tmp_path, """
  struct { int tokens, n_tiles, chunks, want; } calls[] = {
      {1305, 24, 3, 64}, {1305, 24, 32, 64}, {1305, 24, 64, 192}, {1305, 24, 96, 192}, {1540, 20, 16, 64}, {1352, 24, 3, 192}, {929, 36, 3, 192},
      {1085, 36, 96, 192}, {2715, 12, 3, 192}, {31, 3, 3, 64}, {449, 9, 3, 64}, {3585, 36, 3, 128}, {1345, 36, 3, 256}, {48360, 36, 96, 256},
      {16640, 2, 2, 192}, {16449, 2, 2, 192}, {11008, 3, 2, 192}, {33280, 1, 2, 192}};
  for (auto c : calls) {
    const int got = 32 * gemm_token_blocks(c.tokens, c.n_tiles, c.chunks, 256);
    CHECK(got == c.want, "%d tokens, %d tiles, %d chunks: %d", c.tokens, c.n_tiles, c.chunks, got);
  }""")


def test_relay_runs_make_no_round_too_many(tmp_path):
    """Runs follow each other without a gap, are as long as equal shares to a unit, and the longest has no more rounds than of equal shares; where
    those cross a head's end with one unit over on either side (51, 116 and 149 units a head), as many as its units need."""
    _run(tmp_path, """
  for (int wgs = 8; wgs <= 304; wgs += 8)
    for (int heads = 1; heads <= 96; heads += heads < 8 ? 1 : 8)
      for (int per_head = 1; per_head <= 400; per_head += per_head < 160 ? 1 : 17) {
        const int units = heads * per_head;
        if (units <= 4 * wgs) continue;
        for (int fills = 0; fills < 2; ++fills) {
          int most[2] = {0, 0}, at = 0;
          for (int rank = 0; rank < wgs; ++rank) {
            const int begin = relay_cut(rank, units, per_head, wgs, fills), end = relay_cut(rank + 1, units, per_head, wgs, fills);
            CHECK(begin == at && end >= begin && end <= units, "%d x %d units, workgroup %d of %d: [%d, %d)", heads, per_head, rank, wgs, begin, end);
            CHECK(end - begin <= units / wgs + 2 && end - begin >= units / wgs - 1, "%d x %d units, workgroup %d of %d: [%d, %d)", heads, per_head, rank, wgs, begin, end);
            at = end;
            for (int even = 0; even < 2; ++even) {
              int a = even ? (int)((int64_t)rank * units / wgs) : begin, rounds = 0;
              const int b = even ? (int)((int64_t)(rank + 1) * units / wgs) : end;
              for (int part; a < b; a += part) {
                part = (a / per_head + 1) * per_head < b ? (a / per_head + 1) * per_head - a : b - a;
                rounds += relay_rounds(part);
              }
              if (rounds > most[even]) most[even] = rounds;
            }
          }
          CHECK(at == units && most[0] <= most[1], "%d x %d units on %d: %d rounds, %d in equal shares", heads, per_head, wgs, most[0], most[1]);
          if (fills && wgs == 256 && heads == 24 && (per_head == 51 || per_head == 116 || per_head == 149))
            CHECK(most[0] == relay_rounds((units + 255) / 256) && most[1] == most[0] + 1, "%d units: %d and %d rounds", per_head, most[0], most[1]);
          if (!fills && wgs == 256 && heads == 72 && per_head == 16) CHECK(most[0] == 2 && most[1] == 3, "%d and %d rounds", most[0], most[1]);
        }
      }""")


def test_relay_shares_go_by_the_work_of_the_entries(tmp_path):
    """Entries of unequal valid keys, none to 40 tiles of them, shared out among 8 to 304 workgroups: the runs follow each other without a gap from
    the first unit to the last, and no run is longer than the mean by more than two of the longest units (one at either end)."""
    _run(tmp_path, """
  const int tiles[][6] = {{1, 40}, {40, 1}, {5, 5}, {0, 40}, {0, 0}, {1, 2, 4, 8, 16, 40}, {40, 40, 1, 1, 0, 40}, {0, 0, 0, 0, 0, 1}};
  const int entries[] = {2, 6, 70}, workgroups[] = {8, 104, 256, 304}, sizes[] = {1, 3, 24 * 116, 2 * 388, 1030, 16777216};
  for (auto& t : tiles)
    for (int B : entries)
      for (int wgs : workgroups)
        for (int units : sizes) {                                         // of an entry
          auto weight = [&](int b) { return relay_weight(t[b % (B == 2 ? 2 : 6)] * 64); };
          int64_t total = 0, longest = 0;
          for (int b = 0; b < B; ++b) {
            total += weight(b);
            if (weight(b) > longest) longest = weight(b);
          }
          int64_t at = 0;                                                 // units in front of the run
          double done = 0;                                                // ... and their weight, a unit of an entry counting weight(b)
          for (int rank = 0; rank < wgs; ++rank) {
            int64_t end = (int64_t)B * units, before = 0;
            for (int b = 0; b < B; before += weight(b++)) {
              const int64_t into = (int64_t)(rank + 1) * total - before * wgs;
              if (into < 0 || into >= (int64_t)weight(b) * wgs) continue;
              const int unit = relay_unit((int)into, weight(b), wgs, units);
              CHECK(unit >= 0 && unit < units, "unit %d of %d", unit, units);
              end = (int64_t)b * units + unit;
            }
            CHECK(end >= at && end <= (int64_t)B * units, "%d entries x %d units, workgroup %d of %d: [%lld, %lld)", B, units, rank, wgs, (long long)at, (long long)end);
            double run = 0;
            for (int b = 0; b < B; ++b) {
              const int64_t from = at > (int64_t)b * units ? at : (int64_t)b * units, to = end < (int64_t)(b + 1) * units ? end : (int64_t)(b + 1) * units;
              if (to > from) run += (double)(to - from) * weight(b);
            }
            CHECK(run <= (double)total * units / wgs + 2 * longest, "%d entries x %d units: workgroup %d of %d has %g of %g", B, units, rank, wgs, run,
                  (double)total * units);
            done += run, at = end;
          }
          CHECK(at == (int64_t)B * units && done == (double)total * units, "%d entries x %d units: %lld", B, units, (long long)at);
        }""")
