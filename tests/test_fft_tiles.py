"""Column tiles of the FFT passes (xtr_tiles.h, compiled for the host): the handle keeps one choice per precision and
grid for every number of right-hand sides, so what weighs the candidates may only go by the grid. At 75 x 75 x 8 in
complex128 eight right-hand sides have 69 MB of spectra and one has 8.6 MB; the weights are one set."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include "xtr_tiles.h"
int main(int, char **v)
{
    const long long nx = atoll(v[1]), ny = atoll(v[2]), nz = atoll(v[3]);
    const int e = atoi(v[4]), p = 2 * (int)nx;
    for (int t = 0; t < 6; ++t)
        std::printf("%d %.2f\n", xtr::fft_tile_cols(p, e, t), xtr::fft_tile_weight(12 * nx * ny * nz * e, p, e, t));
}
"""


@pytest.fixture(scope="module")
def tiles(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiles")
    (d / "t.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "extreme_amd", "csrc"), "-o", str(d / "t"), str(d / "t.cpp")],
                   check=True)

    def run(nx, ny, nz, e):
        out = subprocess.run([str(d / "t"), *map(str, (nx, ny, nz, e))], check=True, capture_output=True, text=True).stdout
        rows = [line.split() for line in out.splitlines()]
        return [int(r[0]) for r in rows], [float(r[1]) for r in rows]
    return run


# default, narrow, wide, narrow with 512 threads, register, register with the other column count
@pytest.mark.parametrize("grid,e,cols,short", [
    ((30, 30, 64), 16, [16, 16, 16, 16, 16, 16], []),            # 60 points: one tile
    ((64, 64, 32), 16, [16, 8, 32, 8, 16, 32], []),               # 128 points, 25 MB
    ((75, 75, 8), 16, [8, 4, 16, 4, 8, 16], []),                 # 150 points, 8.6 MB
    ((128, 128, 32), 16, [8, 4, 16, 4, 8, 16], [1, 3]),        # 256 points, 101 MB
    ((128, 128, 8), 16, [8, 4, 16, 4, 8, 16], []),                # 25 MB
    ((128, 128, 32), 8, [16, 8, 32, 8, 16, 32], [1, 3]),         # complex64, 50 MB
    ((256, 256, 64), 16, [8, 4, 16, 4, 8, 4], [1, 3, 5]),        # 512 points
])
def test_tiles_of_a_grid(tiles, grid, e, cols, short):
    c, w = tiles(*grid, e)
    assert c == cols
    assert w == [1.1 if t in short else 1.0 for t in range(6)]

