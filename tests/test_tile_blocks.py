"""The share of a 64 x 64 tile that each of its four waves computes (``pycc_amd/csrc/tile_blocks.h``): every 16 x 16
block that holds outputs belongs to exactly one wave, and the rows and columns of LDS that a wave reads for its
blocks lie inside the tile. Compiled for the CPU from the header that the kernel includes."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include "tile_blocks.h"
#include <cstdio>
int main() {
  for (int rb = 1; rb <= 4; ++rb)
    for (int cb = 1; cb <= 4; ++cb) {
      int seen[4][4] = {};
      for (int w = 0; w < 4; ++w) {
        const ccx::WaveBlocks b = ccx::wave_blocks(rb, cb, w);
        const bool form = (b.ni == 0 || b.nj == 0) || (b.ni <= 2 && b.nj <= 2 && b.ni > 0 && b.nj > 0);
        if (!form) return std::printf("%d x %d wave %d: %d x %d blocks\n", rb, cb, w, b.ni, b.nj), 1;
        if (b.ni == 0 || b.nj == 0) continue;   // reads nothing
        if (b.r0 < 0 || b.c0 < 0 || b.r0 + 16 * b.ni > 64 || b.c0 + 16 * b.nj > 64)
          return std::printf("%d x %d wave %d reads rows %d.. columns %d.. past the tile\n", rb, cb, w, b.r0, b.c0), 1;
        for (int i = 0; i < b.ni; ++i)
          for (int j = 0; j < b.nj; ++j) ++seen[b.r0 / 16 + i][b.c0 / 16 + j];
      }
      for (int i = 0; i < 4; ++i)
        for (int j = 0; j < 4; ++j)
          if (seen[i][j] != (i < rb && j < cb)) return std::printf("%d x %d: block %d %d\n", rb, cb, i, j), 1;
    }
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_blocks_of_the_waves(tmp_path):
    src, exe = tmp_path / "blocks.cpp", tmp_path / "blocks"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pycc_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
