"""The prefill GEMM's block-to-tile deal (csrc/es_tiles.hpp, plain C++, compiled
here for the CPU): every tile is one block's, and the XCDs (block b runs on XCD
b % 8) hold equal numbers of blocks, also where the row tiles are not a
multiple of eight. And the rules for the kernel of 256 x 256 tiles, for four weight
rows a wave in the matvec of several token rows, and for the output gate."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "enginesmith-qwen35-08b-long-decode-m5max-round005_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "es_tiles.hpp"
int main(int argc, char** argv) {  // column tiles, row tiles -> the grid's tiles in block order
  const unsigned nb = atoi(argv[1]), mb = atoi(argv[2]);
  for (unsigned b = 0; b < es::gemm_grid(nb, mb); ++b) {
    const es::GemmTile t = es::gemm_tile(b, nb, mb);
    printf("%d %d\n", t.bx, t.by);
  }
}
"""
WIDE = r"""
#include <cstdio>
#include <cstdlib>
#include "es_tiles.hpp"
int main(int argc, char** argv) { printf("%d", (int)es::gemm_wide(atoi(argv[1]), atoi(argv[2]), atoi(argv[3]))); }
"""

ROWS = r"""
#include <cstdio>
#include <cstdlib>
#include "es_tiles.hpp"
int main(int argc, char** argv) { printf("%d", (int)es::qmv_four_rows(atoi(argv[1]) == 1024, atol(argv[2]))); }
"""

GATE = r"""
#include <cstdio>
#include <cstdlib>
#include "es_tiles.hpp"
int main(int argc, char** argv) { printf("%d", (int)es::gate_eight(atoi(argv[1]))); }
"""


def compiled(tmp_path_factory, source):
    d = tmp_path_factory.mktemp("tiles")
    (d / "tiles.cpp").write_text(source)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, "-o", str(d / "tiles"), str(d / "tiles.cpp")], check=True)
    return str(d / "tiles")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    return compiled(tmp_path_factory, PROGRAM)


@pytest.fixture(scope="module")
def wide(tmp_path_factory):
    return compiled(tmp_path_factory, WIDE)


# 56 and 65 column tiles: the MLP's gate/up and the stacked GDN input at 9, 10,
# 17 and 32 tiles of 128 rows; odd and small ones
@pytest.mark.parametrize("nb,mb", [(56, 9), (65, 9), (40, 10), (56, 17), (56, 32), (1, 8), (1, 9), (7, 15), (8, 8),
                                   (13, 23), (28, 9)])
def test_every_tile_once_and_the_xcds_equal(program, nb, mb):
    out = subprocess.run([program, str(nb), str(mb)], check=True, capture_output=True, text=True).stdout
    tiles = np.array(out.split(), int).reshape(-1, 2)
    xcd = np.arange(len(tiles)) % 8
    work = tiles[:, 1] < mb  # a block past the last row tile has none
    tiles, xcd = tiles[work], xcd[work]
    load = np.bincount(xcd, minlength=8)
    assert load.max() - load.min() <= 1, load  # 9 x 56 dealt by whole row tiles: 112 and 56
    assert len(tiles) == nb * mb
    assert len(np.unique(tiles[:, 1] * nb + tiles[:, 0])) == nb * mb
    assert tiles.min() == 0 and tiles[:, 0].max() == nb - 1 and tiles[:, 1].max() == mb - 1
    whole = tiles[:, 1] < mb // 8 * 8  # the tiles dealt a row tile to an XCD
    assert np.array_equal(tiles[whole, 1] % 8, xcd[whole])


# (N, K, rows) on both sides of the rule's lines, and which kernel measured faster
@pytest.mark.parametrize("n,k,m,want", [
    (4096, 3584, 3035, 0), (3584, 3584, 3547, 1), (4096, 3584, 3100, 1), (4096, 3584, 4096, 1), (8192, 4096, 1500, 0),
    (4096, 3584, 7131, 0), (8192, 2048, 3547, 0), (6144, 3584, 5083, 1), (4096, 3584, 11227, 0), (3584, 3584, 13275, 1),
    (6144, 1024, 4096, 0), (4096, 2112, 4096, 0)])
def test_the_kernel_of_256_tiles_takes_what_it_is_faster_at(wide, n, k, m, want):
    out = subprocess.run([wide, str(n), str(k), str(m)], check=True, capture_output=True, text=True).stdout
    assert int(out) == want


# (K, token rows x weight rows) on both sides of the lines, and which form measured faster
@pytest.mark.parametrize("k,outputs,want", [
    (2048, 3072, 0), (2048, 4096, 1), (1536, 5120, 0), (2048, 5120, 0), (2048, 6144, 1), (3584, 11264, 1),
    (1024, 12288, 0), (1024, 18432, 0), (1024, 20480, 0), (1024, 21504, 1), (1024, 32768, 1)])
def test_four_weight_rows_a_wave_where_they_are_faster(tmp_path_factory, k, outputs, want):
    out = subprocess.run([compiled(tmp_path_factory, ROWS), str(k), str(outputs)], check=True, capture_output=True,
                         text=True).stdout
    assert int(out) == want


@pytest.mark.parametrize("rows,want", [(1, 0), (64, 0), (160, 0), (203, 1), (4096, 1)])
def test_the_gate_takes_eight_elements_where_they_are_faster(tmp_path_factory, rows, want):
    out = subprocess.run([compiled(tmp_path_factory, GATE), str(rows)], check=True, capture_output=True, text=True).stdout
    assert int(out) == want
