"""CPU checks of the FAS solver's launch arithmetic (proto_amd/csrc/pm_fas_grid.hpp,
plain C++): what the norm kernel launches against the partials that are held."""
import os
import subprocess

import pytest

import util

PROGRAM = r"""
#include <cstdio>
#include "pm_fas_grid.hpp"
int main()
{
    int b[3];
    long n;
    while (std::scanf("%d %d %d %ld", b, b + 1, b + 2, &n) == 4) {
        const pm::FzGrid g = pm::fz_grid(b, n);
        std::printf("%d %d %u %u %u\n", (int)pm::fz_box(b), g.zc, g.blocks, pm::fas_norm_blocks(b, n),
                    pm::fas_blocks((long)b[0] * b[1] * b[2]));
    }
}
"""


@pytest.fixture(scope="module")
def grids(tmp_path_factory):
    d = tmp_path_factory.mktemp("fas_grid")
    src, exe = str(d / "grid.cpp"), str(d / "grid")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(util.ROOT, "proto_amd", "csrc"), src, "-o", exe],
                   check=True)

    def run(boxes):
        text = "".join("%d %d %d %d\n" % b for b in boxes)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split("\n")
        return [tuple(int(v) for v in line.split()) for line in out if line]
    return run


def boxes():
    sides = [2, 8, 9, 15, 16, 17, 24, 32, 40, 48, 56, 64, 65, 96, 128, 192, 256, 320, 384, 512]
    return [(x, y, z, n) for x in (2, 16, 31, 32, 33, 48, 63, 64, 65) for y in sides for z in sides for n in (1, 2, 8, 27, 512)]


def test_norm_partials_cover_the_launch(grids):
    """The z-marching norm kernel writes one partial per workgroup; a single box of
    unequal extents launches more than the 1024 a per-cell kernel stops at."""
    todo = boxes()
    most = 0
    for (x, y, z, n), (fz, zc, blocks, held, cellwise) in zip(todo, grids(todo)):
        if not fz:
            assert held == cellwise
            continue
        tile = 16 if x <= 32 else 8
        launched = -(-y // tile) * -(-z // zc)
        assert blocks == launched <= held, (x, y, z, n)
        most = max(most, launched / cellwise)
    assert most > 1  # boxes whose launch outgrows the per-cell count are among them
    assert grids([(64, 320, 128, 1), (64, 256, 512, 1)]) == [(1, 4, 1280, 1280, 1024), (1, 8, 2048, 2048, 1024)]
