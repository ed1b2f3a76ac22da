"""CPU check of the LIF scan over runs of rows: with the kernel's own index arithmetic
(csrc/lif_rows.h, compiled for the host) every load of every thread lies in the
plane, and the columns the threads keep are the plane's, each once."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <algorithm>
#include <vector>
#include "lif_rows.h"
using namespace hses;
static bool plane_ok(int64_t rows, int32_t h, int32_t rb) {
    const int64_t plane = rows * h;
    std::vector<int> kept(plane, 0);
    for (int64_t row0 = 0; row0 < rows; row0 += rb) {
        const int32_t here = (int32_t)std::min<int64_t>(rb, rows - row0);
        for (int32_t tid = 0; tid < lif_rows_threads(rb, h); ++tid) {
            const LifCols c = lif_rows_cols(row0, here, h, tid, plane);
            if (c.e < 0 || c.e + 4 > plane) {
                printf("rows %ld h %d row0 %ld tid %d loads [%ld, %ld) of %ld\n", (long)rows, h, (long)row0,
                       tid, (long)c.e, (long)c.e + 4, (long)plane);
                return false;
            }
            if (c.own > 0)
                for (int i = c.over; i < 4; ++i) ++kept[c.e + i];
        }
    }
    for (int k : kept)
        if (k != 1) return printf("rows %ld h %d: a column is kept %d times\n", (long)rows, h, k), false;
    return true;
}
int main(int, char** argv) {
    const int32_t h = atoi(argv[1]), rb = lif_rows_block(h);
    if (!rb || lif_rows_threads(rb, h) > kLifRowsThreads) return rb != 0;
    for (int64_t rows = (4 + h - 1) / h; rows <= 2 * rb + 4; ++rows)
        if (!plane_ok(rows, h, rb)) return 1;
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("lif_rows")
    (d / "bounds.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "hyperscalees_amd", "csrc"),
                    str(d / "bounds.cpp"), "-o", str(d / "bounds")], check=True)
    return str(d / "bounds")


@pytest.mark.parametrize("h", [1, 2, 3, 4, 5, 6, 7, 10, 17, 63, 65, 100, 130, 255, 500, 511, 512, 513])
def test_every_load_lies_in_the_plane(program, h):
    """Every row count up to two blocks and a bit (h 1..3: last blocks of fewer than
    four columns)."""
    r = subprocess.run([program, str(h)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
