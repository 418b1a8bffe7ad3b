"""The token tile of the vectorised conv (csrc/conv_tile.hpp): the shortest
with which all blocks run at once, for any number of channel slabs."""

import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "logssms_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include "conv_tile.hpp"
int main() {
  for (int per_cu = 3; per_cu <= 4; ++per_cu)
    for (int64_t slabs = 1; slabs <= 1100; slabs += slabs < 12 ? 1 : 97)
      for (int64_t t = 1; t < 50000; t += t < 3000 ? 1 : 61) {
        const int tile = gdn::conv_tile(t, slabs, per_cu);
        auto fits = [&](int n) { return (t + n - 1) / n * slabs <= 256 * per_cu; };
        const int shorter = tile > 4 ? tile - 4 : 2;
        const bool whole = tile == 2 || (tile >= 4 && tile <= 32 && tile % 4 == 0);
        if (!whole || (tile < 32 && !fits(tile)) || (tile > 2 && fits(shorter))) {
          std::printf("tokens %lld, slabs %lld, %d blocks a CU: tile %d\n", (long long)t, (long long)slabs, per_cu, tile);
          return 1;
        }
      }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_tile_is_the_shortest_that_runs_in_one_round(tmp_path):
    src, exe = tmp_path / "tile.cpp", tmp_path / "tile"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
