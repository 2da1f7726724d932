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


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_parts_in_fours(tmp_path):
    """With `fours` the same holds; a context of several parts never has fewer than without, a number that `parts` allows is whole fours unless the last ones would be
    empty, and one of a single part stays so."""
    source = SOURCE.replace("nvl_few_split(tiles, part_tiles, parts), per", "nvl_few_split(tiles, part_tiles, parts, true), plain = nvl_few_split(tiles, part_tiles, parts), per")
    source = source.replace("if (n < 1 ||", "if (n < plain) empty += 1; if ((plain == 1) != (n == 1)) empty += 1; if (n > 1 && n % 4 && (n + 3) / 4 * 4 <= parts && "
                            "(tiles + (n + 3) / 4 * 4 - 1) / ((n + 3) / 4 * 4) != per) empty += 1;\n        if (n < 1 ||")
    assert source.count(", true)") == 1 and source.count("plain") == 3
    src, exe = tmp_path / "fours.cpp", tmp_path / "fours"
    src.write_text(source)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout


def test_open_parts_have_room():
    """The parts of a step (their results, two numbers each) and the single parts' rows lie in the step's workspace, whatever its longest context."""
    from nano_vllm_amd import ops
    for hkv, hq in ((8, 16), (1, 16), (2, 4), (4, 20), (8, 24), (16, 32)):
        for b in (1, 2, 3, 4):
            for longest in list(range(1, 2100, 1 if hkv == 8 else 7)) + [4096, 4097, 8192, 16383, 16384]:
                room = ops.paged_attn_decode_workspace_bytes(b, hq, longest)
                for fours in (False, True):
                    parts = ops.open_parts(b, hkv, longest, fours)
                    assert parts >= 1 and b * hq * (parts * 130 * 4 + 128 * 2) <= room, (hkv, hq, b, longest, fours, parts)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_the_split_is_the_documented_one(tmp_path):
    """The text of include/nvl.h, worked out here, against the function that both kernels call."""
    src, exe = tmp_path / "said.cpp", tmp_path / "said"
    src.write_text('#include <cstdio>\n#include "few_split.h"\nint main() {\n  for (int fours = 0; fours < 2; ++fours)\n    for (int parts = 1; parts <= 64; ++parts)\n'
                   '      for (int t = 0; t <= 600; ++t) std::printf("%d\\n", nvl_few_split(t, NVL_OPEN_PART_TILES, parts, fours));\n}\n')
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    told = map(int, subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split())
    up = lambda a, b: -(-a // b)
    for parts in range(1, 65):
        for t in range(601):
            n = max(1, up(t, 8))
            assert next(told) == (n if n <= parts else up(t, up(t, parts))), (t, parts)
    for parts in range(1, 65):
        for t in range(601):
            n = up(t, 8)
            r = up(n, 4) * 4
            assert next(told) == (1 if n <= 1 else n if r == n <= parts else up(t, up(t, min(r, parts)))), (t, parts)
