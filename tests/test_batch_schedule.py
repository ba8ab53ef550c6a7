"""Schedules of batched solves (pict_schedule.hpp), compiled for the host: the longest solve comes first by its time, not by
its iterations, every system has all its jobs once, and the lists follow one order of the systems (no deadlock)."""
import os
import subprocess

import pytest

from pict_amd import build

PROGRAM = r"""
#include <cstdio>
#include "pict_schedule.hpp"
using namespace pict;
int main() {
    // rows, rows per thread (0: one workgroup), workgroups, iterations: 800 short iterations take less than 300 long ones
    const std::vector<int> n{900, 60000, 1900, 30000, 62000}, rpt{0, 8, 0, 4, 8}, nwg{1, 15, 1, 15, 16};
    const std::vector<double> it{800, 300, 500, 280, 310};
    std::vector<unsigned> off, jobs;
    const auto us = block_job_costs(n, rpt, it);
    const double makespan = list_schedule(5, nwg, 20, us, off, jobs);
    printf("%.1f\n", makespan);
    for (double u : us) printf("%.1f ", u);
    printf("\n");
    for (unsigned g = 0; g < 20; ++g) {
        for (unsigned j = off[g]; j < off[g + 1]; ++j) printf("%u:%u ", jobs[j] >> 16, jobs[j] & 0xffffu);
        printf("\n");
    }
}
"""


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")
def test_lists_follow_the_time_of_the_solves(tmp_path):
    (tmp_path / "s.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", build.CSRC, "s.cpp", "-o", "s"], cwd=tmp_path, check=True)
    out = subprocess.run(["./s"], cwd=tmp_path, check=True, capture_output=True, text=True).stdout.splitlines()
    makespan, us = float(out[0]), [float(v) for v in out[1].split()]
    lists = [[tuple(int(x) for x in j.split(":")) for j in ln.split()] for ln in out[2:]]
    order = sorted(range(5), key=lambda s: -us[s])
    assert order == [4, 1, 0, 2, 3] and us[0] > us[2]  # by iterations alone: 0, 2, 4, 1, 3
    assert sorted(j for ln in lists for j in ln) == sorted((s, k) for s, w in enumerate([1, 15, 1, 15, 16]) for k in range(w))
    for ln in lists:
        ranks = [order.index(s) for s, _ in ln]
        assert ranks == sorted(ranks)
    assert lists[0][0][0] == 4 and makespan >= us[4] + us[1]
