"""Which form of the FP32 smoother leg a level takes (sp_legs.h, host
arithmetic): compiled by itself and asked for the sizes that were measured on
both sides of the rule, none of which decides by its columns alone."""

import os
import subprocess

import pytest

from simcoflow3d_amd._paths import PKG_DIR
from tests import test_gpu_smoother_tiles as tiles

PROGRAM = r"""
#include <cstdio>
#include "sp_legs.h"
int main() {
  int nx, ny, nz, sweeps;
  while (std::scanf("%d %d %d %d", &nx, &ny, &nz, &sweeps) == 4) {
    const int h = 2 * sweeps;
    const sp::LegGrid g = sp::leg_grid(nx, ny, nz, 40 - 2 * h, 24 - 2 * h, h, 256);
    std::printf("%d %d %d\n", sp::four_cell_leg(nx, ny, nz, sweeps, 256) ? 4 : 1, g.kchunk, g.gz);
  }
}
"""

# (size, sweeps): four cells per thread measured at least 2 % faster, slower
FOUR = [((256, 256, 256), 2), ((192, 192, 192), 2), ((1024, 1024, 8), 2), ((512, 512, 16), 2),
        ((64, 64, 1024), 2), ((128, 128, 512), 2), ((126, 126, 126), 2), ((99, 101, 103), 2),
        ((97, 130, 75), 2), ((108, 108, 300), 2), ((123, 77, 311), 2), ((152, 152, 152), 1),
        ((128, 128, 64), 1), ((112, 112, 112), 1), ((64, 64, 512), 1)]
ONE = [((256, 256, 8), 2), ((256, 256, 32), 2), ((128, 128, 128), 2), ((160, 160, 160), 2),
       ((640, 160, 10), 2), ((88, 264, 24), 2), ((64, 64, 64), 2), ((112, 112, 112), 2),
       ((135, 141, 60), 2), ((30, 400, 30), 2), ((600, 600, 20), 1), ((132, 124, 40), 1),
       ((144, 144, 144), 1), ((88, 264, 24), 1)]


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    d = tmp_path_factory.mktemp("legs")
    (d / "legs.cpp").write_text(PROGRAM)
    exe = str(d / "legs")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(PKG_DIR, "csrc", "engine"),
                    "-o", exe, str(d / "legs.cpp")], check=True)

    def run(cases):
        text = "".join(f"{s[0]} {s[1]} {s[2]} {w}\n" for s, w in cases)
        r = subprocess.run([exe], input=text, capture_output=True, text=True, check=True, timeout=60)
        return [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    return run


def test_measured_sizes_take_the_faster_form(ask):
    assert [c for c, r in zip(FOUR, ask(FOUR)) if r[0] != 4] == []
    assert [c for c, r in zip(ONE, ask(ONE)) if r[0] != 1] == []


def test_sizes_of_the_tile_tests(ask):
    """The GPU tests of the legs reach the form that they are meant for."""
    four = [(s, w) for s in tiles.FOUR for w in (1, 2)]
    four += [(s, 1) for s in tiles.FOUR_1] + [(s, 2) for s in tiles.FOUR_2]
    assert [c for c, r in zip(four, ask(four)) if r[0] != 4] == []
    assert {s[0] % 4 for s, w in four if w == 2} == {s[0] % 4 for s, w in four if w == 1} == {0, 1, 2, 3}
    one = [(s, w) for s in tiles.SIZES for w in (1, 2)]
    assert [c for c, r in zip(one, ask(one)) if r[0] != 1] == []


def test_chunks_cover_the_planes(ask):
    cases = [((40, 40, nz), w) for nz in list(range(1, 40)) + [255, 256, 257] for w in (1, 2)]
    for (size, _), (_, chunk, gz) in zip(cases, ask(cases)):
        assert chunk > 0 and chunk % 2 == 0 and (gz - 1) * chunk < size[2] <= gz * chunk
