"""The tile of grid points a wave of the exact assignment takes
(tess2_amd/csrc/owner_tiles.hpp), on the host: a wave never meets more than a
few hundred particles one after the other however coarse the grid is, its points
are a power-of-two box that fits the lanes, and tiles stay countable."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "tess2_amd", "csrc")

HARNESS = r"""
#include <cmath>
#include <cstdio>
#include <initializer_list>
#include "owner_tiles.hpp"
using namespace t2;

static int bad = 0;
static void check(const int d[3], const double s[3], const int b[3])
{
    const OwnerTile t = owner_tile(d, s, b);
    const int bits = t.bits[0] + t.bits[1] + t.bits[2];
    double tiles = 1.0;
    for (int a = 0; a < 3; ++a) tiles *= ((d[a] - 1) >> t.bits[a]) + 1;
    // particles one lane meets in a row
    const double row = tile_meets(t, s, b) * t.points / 64.0;
    if ((1 << bits) != t.points || (t.points != 64 && t.points != 8 && t.points != 1) ||
        tiles > 2147483000.0 || row > 400.0) {
        ++bad;
        std::printf("%d x %d x %d, %g %g %g: %d points (%d %d %d), %g tiles, %g in a row\n", d[0],
                    d[1], d[2], s[0], s[1], s[2], t.points, t.bits[0], t.bits[1], t.bits[2], tiles,
                    row);
    }
}

int main()
{
    const int g[] = {1, 2, 3, 5, 9, 17, 33, 65, 129, 257, 700};
    for (double particles : {1.0, 1e3, 262e3, 2e6, 3e8})
        for (int x : g)
            for (int y : g)
                for (int z : g) {
                    const int d[3] = {x, y, z};
                    const double side = std::cbrt(particles);
                    const double s[3] = {side / (x > 1 ? x - 1 : 1), side / (y > 1 ? y - 1 : 1),
                                         side / (z > 1 ? z - 1 : 1)};
                    // grids of points as dense as the memory of a few runs
                    if ((double)x * y * z * 64.0 < particles && x < 9 && particles > 1e8) continue;
                    const int b[3] = {(int)side + 1, (int)side + 1, (int)side + 1};
                    check(d, s, b);
                }
    const int huge[3] = {2000, 2000, 2000};
    const double coarse[3] = {30.0, 30.0, 30.0};
    const int many[3] = {60000, 60000, 60000};
    const OwnerTile t = owner_tile(huge, coarse, many);     // 8e9 points
    if (t.points != 64) ++bad;
    // a fine grid keeps 64 points a wave, in a cube
    const int fine[3] = {192, 192, 192};
    const double f[3] = {0.33, 0.33, 0.33};
    const int side[3] = {64, 64, 64};
    const OwnerTile c = owner_tile(fine, f, side);
    if (c.points != 64 || c.bits[0] != 2 || c.bits[1] != 2 || c.bits[2] != 2) ++bad;
    // and so does one whose particles all lie in a small part of it
    const int wide[3] = {257, 257, 257}, ten[3] = {11, 11, 11};
    const double w[3] = {3.9, 3.9, 3.9};
    if (owner_tile(wide, w, ten).points != 64) ++bad;
    return bad;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ missing")
def test_tiles_are_bounded(tmp_path):
    src = tmp_path / "tiles.cpp"
    src.write_text(HARNESS)
    exe = tmp_path / "tiles"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:2000]
