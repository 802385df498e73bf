"""The division by a reciprocal with which the gather kernels find their block
of columns and chunk of layers: compiled for the host and compared with / and %
for rows of one block (a grid of at most 256 columns or edges), of two, three
and odd counts, powers of two and the largest grids', over every linear index
near 0, near multiples of the row and near the largest."""
import os
import subprocess

import pytest

from conftest import ROOT
from game_archived_amd.build import HIPCC

PROGRAM = r"""
#include <stdio.h>
#include "rkhevi_dev.h"
int main()
{
    const unsigned rows[] = {1, 2, 3, 5, 7, 8, 11, 41, 64, 121, 255, 256, 640, 641, 1921, 7681, 10240, 30721, 122881};
    long long n = 0, bad = 0;
    for (unsigned gx : rows) {
        for (int cells : {(int)(gx - 1)*TPB + 1, (int)gx*TPB}) {
            const Span sp = span_of(cells, 26, 9);
            auto check = [&](unsigned m) {
                const Blk b = block_at(m, gx, sp.rcp);
                ++n;
                if (b.x != m%gx || b.y != m/gx) {
                    if (bad++ < 5) printf("row of %u blocks, index %u: (%u, %u), not (%u, %u)\n", gx, m, b.x, b.y, m%gx, m/gx);
                }
            };
            for (unsigned m = 0; m < 200000; ++m) check(m);
            for (unsigned q = 1; q < 4000; ++q)
                for (int k = -2; k <= 2; ++k) {
                    const long long m = (long long)q*(4294967295u/4000)/gx*gx + k;
                    if (m >= 0 && m <= 4294967295LL) check((unsigned)m);
                }
            for (unsigned k = 0; k < 2000; ++k) check(4294967295u - k);
        }
    }
    printf("%lld indexes, %lld wrong\n", n, bad);
    return bad != 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs the HIP compiler (host pass only)")
def test_block_of_a_linear_index(tmp_path):
    src = tmp_path / "block_map.hip"
    src.write_text(PROGRAM)
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-host-only", "-Wno-unused-function", "-I",
                    os.path.join(ROOT, "game_archived_amd", "csrc"), "-o", str(tmp_path / "block_map"), str(src)], check=True)
    r = subprocess.run([str(tmp_path / "block_map")], stdout=subprocess.PIPE, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
