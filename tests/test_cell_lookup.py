"""The broadphase cell of a point, which the engine finds with a reciprocal and
one residual step (state.h: overCell), is the one that the division gives.

The engine's own headers are compiled for the host.  The quotient may differ
from the division's in the last place (where, the program counts), so only a
float next to a cell's edge could fall into another cell: those are all
visited, 4,096 floats to either side of every edge, and a sample of the range
shows that no quotient is off by more.  With the argument "all" the program
visits every float in [0, 1e5], in two minutes; all cells agree there too.
"""
from __future__ import annotations

import os
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "carl_amd" / "csrc"
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))

PROGRAM = r"""
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include "state.h"
using namespace carl;

static float at(uint32_t bits) { float f; memcpy(&f, &bits, 4); return f; }
static uint32_t bitsOf(float f) { uint32_t b; memcpy(&b, &f, 4); return b; }

static long cellsOff = 0, lastPlace = 0, further = 0, visited = 0;
static void visit(float x, float c, float cells)
{
    const float q = overCell(x, c), d = x / c;
    visited++;
    const int off = std::abs((int)(bitsOf(q) - bitsOf(d)));
    lastPlace += off == 1;
    further += off > 1;
    cellsOff += (int)fmin_(q, cells - 1.f) != (int)fmin_(d, cells - 1.f);
}

// the cells as three divisions give them
static void divided(V3 p, int* out)
{
    const float v[3] = { (p.x - kArenaMin.x) / kCellX, (p.y - kArenaMin.y) / kCellY, (p.z - kArenaMin.z) / kCellZ };
    const float n[3] = { 48.f, 48.f, 10.f };
    for (int k = 0; k < 3; k++) out[k] = (int)fmin_(fmax_(v[k], 0.f), n[k] - 1.f);
}

int main(int argc, char**)
{
    const uint32_t end = bitsOf(1e5f), step = argc > 1 ? 1 : 251;
    const float size[3] = { kCellX, kCellY, kCellZ }, cells[3] = { 48.f, 48.f, 10.f };
    for (int k = 0; k < 3; k++) {
        cellsOff = lastPlace = further = visited = 0;
        for (uint32_t b = 0; b <= end; b += step) visit(at(b), size[k], cells[k]);
        for (int e = 0; e <= (int)cells[k] + 1; e++) {
            const uint32_t edge = bitsOf((float)e * size[k]);
            for (int i = -4096; i <= 4096; i++)
                if ((int)edge + i >= 0) visit(at(edge + i), size[k], cells[k]);
        }
        printf("size %.9g visited %ld last place %ld further %ld cells %ld\n", size[k], visited, lastPlace, further, cellsOff);
    }
    // whole points: inside, at the bounds, beyond them and not finite
    const float inf = std::numeric_limits<float>::infinity(), nan = std::numeric_limits<float>::quiet_NaN();
    const float odd[] = { 0.f, -0.f, 1e-40f, -1e-40f, 99999.f, 100001.f, -1e5f, 3e38f, -3e38f, inf, -inf, nan };
    long points = 0, wrong = 0;
    auto point = [&](V3 p) {
        int c[3], d[3];
        cellOf(p, c[0], c[1], c[2]);
        divided(p, d);
        points++;
        wrong += memcmp(c, d, sizeof c) != 0;
    };
    for (float x : odd) for (float y : odd) for (float z : odd) point(V3{ x, y, z });
    uint64_t s = 1;
    auto uniform = [&](float lo, float hi) {
        s = s * 6364136223846793005ull + 1442695040888963407ull;
        return lo + (hi - lo) * (float)(s >> 40) * 0x1p-24f;
    };
    for (int i = 0; i < 1000000; i++) point(V3{ uniform(-5000.f, 5000.f), uniform(-7000.f, 7000.f), uniform(-500.f, 2600.f) });
    printf("points %ld wrong %ld\n", points, wrong);
    return 0;
}
"""


@pytest.fixture(scope="module")
def report(tmp_path_factory):
    where = tmp_path_factory.mktemp("cells")
    (where / "cells.hip").write_text(PROGRAM)
    subprocess.run([str(ROCM / "bin" / "hipcc"), "--offload-arch=gfx950", "--offload-host-only", "-O2", "-std=c++17",
                    "-ffp-contract=off", "-Wno-unused-function", f"-I{CSRC}", str(where / "cells.hip"), "-o",
                    str(where / "cells")], check=True)
    out = subprocess.run([str(where / "cells")], check=True, capture_output=True, text=True).stdout
    return [line.split() for line in out.splitlines()]


def test_every_float_near_an_edge_falls_into_the_division_s_cell(report):
    assert len(report) == 4
    for words in report[:3]:
        counts = dict(zip(("visited", "last place", "further", "cells"), map(int, (words[3], words[6], words[8], words[10]))))
        assert counts["visited"] > 4_000_000
        assert counts["further"] == 0 and counts["cells"] == 0, words


def test_points_outside_the_grid_are_clamped_alike(report):
    words = report[3]
    assert int(words[1]) > 1_000_000 and int(words[3]) == 0, words
