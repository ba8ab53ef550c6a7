"""Placement of a system's rows on the workgroups of the on-chip solvers (pict_block.hpp): every row has one position and
every position at most one row, for rows in order, blocks of lines, and lines cut into strips.  The functions are compiled
for the host; no GPU is needed."""
import os
import subprocess

import pytest

from pict_amd import build

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "pict_block.hpp"
using namespace pict;
template <int C, int NZ>
static int check(int argc, char **v) {
    BlockMap m{};
    m.n = atoi(v[2]), m.brick = atoi(v[3]), m.line = atoi(v[4]), m.ny = atoi(v[5]);
    const int nz = atoi(v[6]);
    m.strips = atoi(v[7]), m.a = atoi(v[8]), m.b = atoi(v[9]);
    m.nx = m.strips > 1 ? ((m.line + m.strips - 1) / m.strips + 7) / 8 * 8 : m.line;
    m.nby = m.brick ? (m.ny + m.a - 1) / m.a : 1;
    const int nbz = m.brick ? (nz + m.b - 1) / m.b : 1;
    m.lines = m.brick ? m.ny * nbz * m.b : m.ny * nz;
    m.nz = m.strips * nbz * m.b;
    m.nwg = m.brick ? m.strips * m.nby * nbz : (int)(((long long)m.strips * m.lines * m.nx + C - 1) / C);
    m.inx = 1.0f / m.nx, m.iny = 1.0f / m.ny, m.ia = 1.0f / m.a, m.ib = 1.0f / m.b, m.inby = 1.0f / m.nby;
    m.iline = 1.0f / m.line, m.ilines = 1.0f / m.lines;
    if (!m.brick && m.strips == 1) m = whole_map(m.n, (m.n + C - 1) / C);
    if ((long long)m.nwg * C >= 1 << 21 || (m.brick && m.nx * m.a * m.b > C)) return 3;
    std::vector<char> seen(m.n, 0);
    long long rows = 0;
    for (int bid = 0; bid < m.nwg; ++bid)
        for (int li = 0; li < C; ++li) {
            const int i = block_row<C, NZ>(m, bid, li);
            if (i < 0) continue;
            if (i >= m.n || seen[i]++ || block_pos<C, NZ>(m, i) != (unsigned)(bid * C + li)) return 1;
            ++rows;
        }
    return rows == m.n ? 0 : 2;
}
int main(int argc, char **v) {
    const int C = atoi(v[1]);
    if (!atoi(v[3])) return C == 512 ? check<512, 5>(argc, v) : check<4096, 5>(argc, v);
    return C == 512 ? check<512, 7>(argc, v) : C == 4096 ? check<4096, 7>(argc, v) : check<7168, 7>(argc, v);
}
"""

CASES = [
    # C, n, brick, line, ny, nz, strips, a, b
    (512, 30000, 0, 300, 100, 1, 1, 1, 1),
    (4096, 1048573, 0, 300, 100, 1, 1, 1, 1),
    (512, 2049, 0, 300, 100, 1, 1, 1, 1),
    (512, 449 * 70, 0, 449, 70, 1, 3, 1, 1),
    (512, 449 * 70 - 13, 0, 449, 70, 1, 3, 1, 1),
    (4096, 1000 * 1000, 0, 1000, 1000, 1, 2, 1, 1),
    (4096, 1023 * 1021, 0, 1023, 1021, 1, 7, 1, 1),
    (512, 24 * 17 * 16, 1, 24, 17, 16, 1, 3, 6),
    (7168, 192 * 96 * 96, 1, 192, 96, 96, 1, 6, 6),
    (7168, 192 * 96 * 96 - 5000, 1, 192, 96, 96, 1, 7, 5),
    (512, 400 * 10 * 9, 1, 400, 10, 9, 2, 2, 1),
    (4096, 1000 * 9 * 8, 1, 1000, 9, 8, 8, 4, 2),
    (7168, 512 * 48 * 40, 1, 512, 48, 40, 4, 8, 7),
    (7168, 512 * 48 * 40 - 777, 1, 512, 48, 40, 3, 5, 7),
]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("map")
    (d / "map.hip").write_text(PROGRAM)
    subprocess.run([build.HIPCC, "-O2", "-std=c++17", "--offload-host-only", "-I", build.CSRC, "-c", "map.hip", "-o",
                    "map.o"], cwd=d, check=True)
    subprocess.run([build.HIPCC, "map.o", "-o", "map"], cwd=d, check=True)
    return str(d / "map")


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")
@pytest.mark.parametrize("case", CASES)
def test_rows_and_positions_are_one_to_one(program, case):
    assert subprocess.run([program] + [str(v) for v in case]).returncode == 0
