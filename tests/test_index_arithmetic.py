"""Index arithmetic of the kernels at sizes and ends where it can go wrong, in a host build of the header they share: no GPU needed."""
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
