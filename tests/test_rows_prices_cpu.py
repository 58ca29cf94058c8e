"""Tiles of f32 products of rows, as they are counted out on the host."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# (m, n, k, groups, gated) -> 128 x 128, 64 x 128 or 64 x 64
TILES = {
    # a few tiles are a round like any other: the smallest ones
    (128, 256, 2048, 0, 0): 11, (256, 16, 2048, 0, 0): 11, (200, 128, 1024, 0, 0): 11, (64, 64, 64, 0, 0): 11, (300, 16, 2048, 0, 0): 11, (2, 2, 2048, 0, 0): 11, (100, 128, 2048, 0, 1): 12,
    (64, 64, 2048, 0, 1): 12,
    # one tile past a round is a second one
    (5504, 768, 2048, 0, 0): 11, (5504, 384, 2048, 0, 1): 12,
    # more tile rows than a grid has: the tile that has fewer, up to as many as that one has
    (65535 * 64, 8, 8, 0, 0): 11, (65535 * 64 + 1, 8, 8, 0, 0): 22, (5000000, 8, 8, 0, 0): 22, (65535 * 128, 8, 8, 0, 0): 22, (5000000, 8, 8, 0, 1): 22, (65535 * 64 - 64, 8, 8, 1, 0): 11, (65535 * 64 - 63, 8, 8, 1, 0): 22,
    # as measured: the fuller last round
    (509, 5632, 2048, 0, 1): 12, (1024, 5632, 2048, 0, 1): 22, (509, 10304, 2048, 0, 0): 12, (700, 6592, 2048, 0, 0): 11, (1531, 2048, 2048, 0, 0): 11, (2036, 1408, 2048, 16, 1): 22,
    (1200, 1408, 2048, 16, 1): 12,
}
PROGRAM = r"""
#include "rows_prices.h"

#include <cstdio>

int main() {
  int m, n, k, groups, gated;
  while (scanf("%d %d %d %d %d", &m, &n, &k, &groups, &gated) == 5) printf("%d\n", ughip::f32_rows_tile(m, n, k, groups, gated != 0));
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_f32_rows_take_the_tile_whose_rounds_are_shortest(tmp_path):
    (tmp_path / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "ug_amd", "csrc", "ughip"), str(tmp_path / "main.cpp"), "-o", str(tmp_path / "tiles")], check=True)
    asked = "\n".join(" ".join(map(str, key)) for key in TILES)
    out = subprocess.run([str(tmp_path / "tiles")], input=asked, capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and dict(zip(TILES, map(int, out.stdout.split()))) == TILES
