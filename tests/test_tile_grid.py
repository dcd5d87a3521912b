"""The boxes of the tiled sweeps (tile_grid.h): at most as many as asked for,
near cubes, and nearly all that a device can hold where the boxes are large."""
import os
import subprocess

import pytest

from conftest import ROOT

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include "tile_grid.h"
int main(int argc, char** argv) {
    const int ext[3] = {std::atoi(argv[1]), std::atoi(argv[2]), std::atoi(argv[3])};
    for (int units = 1; units <= 256; ++units)
        for (long long rows : {100ll, 100000ll}) {
            int k[3] = {0, 0, 0};
            astg::tileGrid(units, rows * units, 256, ext, k);
            std::printf("%d %d %d ", k[0], k[1], k[2]);
            astg::tileGrid(units, rows * units, units, ext, k);
            std::printf("%d %d %d\n", k[0], k[1], k[2]);
        }
}
"""


@pytest.fixture(scope="module")
def grids(tmp_path_factory):
    d = tmp_path_factory.mktemp("grid")
    (d / "grid.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I" + os.path.join(ROOT, "ast-grid_amd", "csrc"),
                    str(d / "grid.cpp"), "-o", str(d / "grid")], check=True)

    def run(ext):
        """Per count asked for: few or many rows on a device of 256 units, the
        same on a device of that many units."""
        out = subprocess.run([str(d / "grid")] + [str(e) for e in ext], capture_output=True, text=True, check=True).stdout
        v = [tuple(int(x) for x in line.split()) for line in out.splitlines()]
        return [(a[:3], b[:3], a[3:], b[3:]) for a, b in zip(v[::2], v[1::2])]
    return run


@pytest.mark.parametrize("ext", [(129, 129, 129), (513, 513, 513), (129, 41, 121), (385, 769, 1), (1, 65, 65), (9, 1, 1),
                                 (65, 65, 3)])
def test_boxes(grids, ext):
    axes = [a for a in range(3) if ext[a] > 1]
    for K, (few, many, few_all, many_all) in enumerate(grids(ext), 1):
        for k in (few, many, few_all, many_all):
            assert all(k[a] == 1 for a in range(3) if a not in axes)
            assert 1 <= k[0] * k[1] * k[2] <= K
        assert few_all == few
        if K < 256:
            assert many == few  # not all units asked for
        # a box per unit, large boxes: 8 of 11 is the worst (nine would be a slab, ten a bar)
        assert 8 * K <= 11 * many_all[0] * many_all[1] * many_all[2]
        edges = [ext[a] / many_all[a] for a in axes]
        if K >= 8 and min(ext[a] for a in axes) > 8:
            assert max(edges) <= 2.0 * min(edges)


def test_cubes(grids):
    g = grids((513, 513, 513))
    few = {K: g[K - 1][0] for K in (1, 2, 3, 4, 5, 7, 8, 15, 27, 96, 200, 256)}
    assert {K: k[0] * k[1] * k[2] for K, k in few.items()} == {1: 1, 2: 1, 3: 1, 4: 4, 5: 4, 7: 4, 8: 8, 15: 8, 27: 27,
                                                               96: 80, 200: 180, 256: 216}
    assert g[255][1] in [(6, 6, 7), (6, 7, 6), (7, 6, 6)]
