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


# (m, n, k, groups, gated, lookup) -> rounded ahead of the product, as either was measured (us on the way / ahead)
AHEAD = {
    (2, 64, 64, 0, 1, 0): 0, (2, 64, 512, 0, 1, 0): 1, (2, 64, 2048, 0, 1, 0): 1,                 # 3.3 / 6.2, 6.8 / 5.9, 19.9 / 9.3
    (130, 64, 64, 0, 1, 0): 1, (32, 704, 128, 0, 1, 0): 0,                                        # 6.7 / 5.9, 5.4 / 6.1
    (2, 704, 128, 0, 0, 1): 0, (2, 704, 512, 0, 0, 1): 1, (64, 64, 64, 0, 0, 1): 1,               # 5.0 / 6.0, 7.2 / 5.9, 7.1 / 5.9
    (32, 704, 128, 4, 0, 0): 0, (32, 704, 1024, 4, 0, 0): 1, (64, 64, 64, 64, 0, 0): 1,           # 4.3 / 6.4, 9.1 / 8.2, 9.6 / 6.0
    (16, 2048, 384, 0, 0, 0): 0, (16, 2048, 768, 0, 0, 0): 1, (16, 2048, 1024, 0, 0, 0): 1,       # 5.7 / 6.0, 7.7 / 6.9, 9.1 / 6.7
    (300, 2048, 640, 0, 0, 0): 0, (16, 2048, 320, 16, 1, 0): 0, (16, 5632, 2048, 0, 1, 0): 1,     # 8.0 / 8.8, 9.2 / 13.5, 29.2 / 15.3
    (64, 704, 1024, 16, 1, 0): 1, (64, 1408, 1024, 16, 1, 0): 1, (64, 2048, 1024, 16, 1, 0): 0,   # 17.2 / 12.9, 20.8 / 18.8, 22.7 / 26.9
}
AHEAD_PROGRAM = r"""
#include "rows_prices.h"

#include <cstdio>

int main() {
  int m, n, k, groups, gated, lookup;
  while (scanf("%d %d %d %d %d %d", &m, &n, &k, &groups, &gated, &lookup) == 6) printf("%d\n", ughip::rows_rounded_ahead(m, n, k, groups, gated != 0, lookup != 0));
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_rows_are_rounded_ahead_of_a_product_where_that_pays_for_the_launch(tmp_path):
    (tmp_path / "main.cpp").write_text(AHEAD_PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "ug_amd", "csrc", "ughip"), str(tmp_path / "main.cpp"), "-o", str(tmp_path / "ahead")], check=True)
    asked = "\n".join(" ".join(map(str, key)) for key in AHEAD)
    out = subprocess.run([str(tmp_path / "ahead")], input=asked, capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and dict(zip(AHEAD, map(int, out.stdout.split()))) == AHEAD


# (us on the tiles, us on rows_product, bytes between the tiles and their fold) -> on the tiles
ON_TILES = {
    (771.0, 868.0, 2048 * 11264 * 4): 1, (771.0, 868.0, 1 << 27): 1, (771.0, 868.0, (1 << 27) + 1): 0, (6105.2, 6340.0, 16384 * 11264 * 4): 0, (771.0, 868.0, 0): 1,
    (-1.0, 868.0, 0): 0, (840.0, 868.0, 0): 0,
}
ON_TILES_PROGRAM = r"""
#include "rows_prices.h"

#include <cstdio>

int main() {
  double tiles, other;
  size_t bytes;
  while (scanf("%lf %lf %zu", &tiles, &other, &bytes) == 3) printf("%d\n", ughip::f32_rows_on_tiles(tiles, other, bytes));
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_f32_rows_take_no_more_of_the_devices_block_than_its_share(tmp_path):
    (tmp_path / "main.cpp").write_text(ON_TILES_PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "ug_amd", "csrc", "ughip"), str(tmp_path / "main.cpp"), "-o", str(tmp_path / "on_tiles")], check=True)
    asked = "\n".join(" ".join(map(str, key)) for key in ON_TILES)
    out = subprocess.run([str(tmp_path / "on_tiles")], input=asked, capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and dict(zip(ON_TILES, map(int, out.stdout.split()))) == ON_TILES


# (rows, vdim, CUs) -> results of a workgroup
MERGED = {
    (16, 128, 256): 16, (32, 128, 256): 16, (33, 128, 256): 32, (64, 128, 256): 32, (65, 128, 256): 64, (128, 128, 256): 64, (129, 128, 256): 128, (256, 128, 256): 128, (2048, 128, 256): 128,
    (128, 64, 256): 32, (129, 64, 256): 64, (512, 64, 256): 64, (2048, 16, 256): 16, (2048, 8, 256): 16, (2048, 17, 256): 32, (128, 32, 256): 16, (129, 32, 256): 32, (64, 200, 256): 64, (512, 200, 256): 128,
    (512, 1, 256): 16, (128, 128, 64): 128,
}
MERGED_PROGRAM = r"""
#include "rows_prices.h"

#include <cstdio>

int main() {
  size_t rows, vdim;
  int cus;
  while (scanf("%zu %zu %d", &rows, &vdim, &cus) == 3) printf("%d\n", ughip::latent_merge_results(rows, vdim, cus));
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_latent_merge_leaves_no_cu_idle_and_makes_no_more_than_there_is(tmp_path):
    (tmp_path / "main.cpp").write_text(MERGED_PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "ug_amd", "csrc", "ughip"), str(tmp_path / "main.cpp"), "-o", str(tmp_path / "merged")], check=True)
    asked = "\n".join(" ".join(map(str, key)) for key in MERGED)
    out = subprocess.run([str(tmp_path / "merged")], input=asked, capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and dict(zip(MERGED, map(int, out.stdout.split()))) == MERGED


# (m, n, k) -> us that an f32 product with a lookup takes on the tile it has, as measured; n 5632 and 1024 rows are 352 tiles of 128 x 128, where 64 x 64 would be priced lower
LOOKUPS = {(1024, 5632, 512): 103.4, (1024, 5632, 128): 50.0, (2000, 5632, 128): 74.8, (100, 64, 512): 17.1, (200, 1024, 512): 17.4}
LOOKUPS_PROGRAM = r"""
#include "rows_prices.h"

#include <cstdio>

int main() {
  int m, n, k;
  while (scanf("%d %d %d", &m, &n, &k) == 3) printf("%f\n", ughip::f32_lookup_us(m, n, k));
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_f32_lookups_are_priced_on_the_tile_they_have(tmp_path):
    (tmp_path / "main.cpp").write_text(LOOKUPS_PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "ug_amd", "csrc", "ughip"), str(tmp_path / "main.cpp"), "-o", str(tmp_path / "lookups")], check=True)
    asked = "\n".join(" ".join(map(str, key)) for key in LOOKUPS)
    out = subprocess.run([str(tmp_path / "lookups")], input=asked, capture_output=True, text=True, timeout=60)
    assert out.returncode == 0
    for key, us in zip(LOOKUPS, map(float, out.stdout.split())):
        assert abs(us - LOOKUPS[key]) <= 0.2 * LOOKUPS[key], (key, us)  # a price: what the formula leaves out is within a fifth
