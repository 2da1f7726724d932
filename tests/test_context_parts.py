"""How decode attention of few sequences cuts a context into parts (csrc/few_split.h), enumerated on the host: every tile belongs to one part, no part is empty,
and one part owns the new token, whatever the limit on their number."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano_vllm_amd", "csrc")
# the bounds of a part as decode_few_kernel has them
SOURCE = """
#include <cstdio>
#include <initializer_list>
#include "few_split.h"
int main() {
  for (int part_tiles : {8, 32})
    for (int parts = 1; parts <= 64; ++parts)
      for (int tiles = 1; tiles <= 1100; ++tiles) {
        const int n = nvl_few_split(tiles, part_tiles, parts), per = nvl_few_div(tiles, n);
        int next = 0, owners = 0, empty = 0;
        for (int p = 0; p < n; ++p) {
          const int t0 = p * per, t1 = tiles < t0 + per ? tiles : t0 + per;
          empty += t0 >= t1;
          owners += t1 == tiles;
          if (t0 != next) empty += 1000;
          next = t1;
        }
        if (n < 1 || n > parts || empty || owners != 1 || next != tiles) {
          std::printf("%d tiles in parts of %d, up to %d: %d parts, %d empty, %d own the new token\\n", tiles, part_tiles, parts, n, empty, owners);
          return 1;
        }
      }
  for (int b = 1; b <= 256; ++b)
    for (int a = 1; a < (1 << 20); a += a < 5000 ? 1 : 97)
      if (nvl_few_div(a, b) != (a + b - 1) / b) return 3;
  return nvl_few_split(0, 8, 16) == 1 ? 0 : 2;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_every_tile_and_the_new_token_belong_to_one_part(tmp_path):
    src, exe = tmp_path / "split.cpp", tmp_path / "split"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
