"""How the MFMA grouped GEMM cuts an expert's rows into tiles (csrc/include/eia_moe_tiles.h, as the host
compiler sees it)."""

import os
import shutil
import subprocess

import pytest

INCLUDE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "csrc", "include")
MAIN = """
#include "eia_moe_tiles.h"
#include <cstdio>
int main() {
  for (int whole = 0; whole < 2; ++whole)
    for (int max_mu = 1; max_mu <= 5; ++max_mu)
      for (int rows = 1; rows <= 1500; ++rows) {
        const int tiles = moe_slice_tiles(rows, max_mu);
        for (int t = 0; t < tiles; ++t) {
          const MoeTile m = moe_slice_tile(rows, tiles, t, whole, max_mu);
          std::printf("%d %d %d %d %d\\n", whole, max_mu, rows, m.lo, m.mu);
        }
      }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_every_row_lies_in_one_tile(tmp_path):
    src, exe = tmp_path / "tiles.cpp", tmp_path / "tiles"
    src.write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", INCLUDE, str(src), "-o", str(exe)], check=True)
    slices = {}
    for line in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines():
        whole, max_mu, rows, lo, mu = map(int, line.split())
        slices.setdefault((whole, max_mu, rows), []).append((lo, mu))
    assert len(slices) == 2 * 5 * 1500
    for (whole, max_mu, rows), tiles in slices.items():
        at = 0
        for lo, mu in tiles:
            assert lo == at and 1 <= mu <= max_mu, (whole, max_mu, rows, tiles)
            at += mu
        units = -(-rows // 64)
        assert len(tiles) == -(-units // max_mu)
        assert units <= at < units + max_mu if whole else at == units
