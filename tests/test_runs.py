"""Runs of entries per workgroup with lengths up to the largest int (kron_runs.hpp): no run begins before the batch or
past it, every entry is in exactly one, and the kernels take their runs from there."""
import os
import re
import subprocess

import numpy as np
import pytest

import oracle
from helpers import accumulation_bound
from kronmult993_amd import api, workloads as W
from kronmult993_amd.device import DeviceBatch

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kronmult993_amd", "csrc")
INT_MAX = 2 ** 31 - 1

CHECK = r"""
#include "kron_runs.hpp"
#include <climits>
#include <cstdio>
int main()
{
    int const nbs[] = {1, 7, 333, 4096, 306783379, 400000000, INT_MAX - 1, INT_MAX};
    long const lens[] = {1, 5, 64, 400000000, INT_MAX, 4l * INT_MAX};
    for (int nb : nbs)
        for (long len : lens)
        {
            long const runs = kronruns::count(nb, len), grid = (runs + 7) / 8 * 8;
            if (grid > 1 << 16) continue;
            long covered = 0;
            for (long i = 0; i < grid; ++i)
            {
                int const b = kronruns::begin(i, len, nb), e = kronruns::end(b, len, nb);
                if (b != (covered < nb ? covered : nb) || e < b || e > nb) return std::printf("nb %d len %ld run %ld: [%d, %d)\n", nb, len, i, b, e), 1;
                covered += e - b;
            }
            if (covered != nb) return std::printf("nb %d len %ld: %ld entries\n", nb, len, covered), 1;
        }
    return 0;
}
"""


def test_run_bounds(tmp_path):
    src, exe = tmp_path / "runs.cpp", tmp_path / "runs"
    src.write_text(CHECK)
    subprocess.run(["g++", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-I", CSRC, "-o", str(exe),
                    str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr


def test_kernels_form_no_start_in_32_bits():
    for name in sorted(os.listdir(CSRC)):
        with open(os.path.join(CSRC, name)) as f:
            assert not re.search(r"xcd_run_index\(\)\s*\*", f.read()), name


@pytest.mark.parametrize("d,n,itemsize,family", [(6, 4, 8, api.FAMILY_REGISTER), (4, 8, 8, api.FAMILY_REGISTER),
                                                 (6, 4, 8, api.FAMILY_MATRIX), (3, 4, 4, api.FAMILY_WAVE),
                                                 (5, 3, 8, api.FAMILY_WAVE)])
def test_grid_of_longest_run(d, n, itemsize, family):
    info = api.launch_info(d, n, itemsize, 400000000, {"family": family, "entries_per_workgroup": INT_MAX})
    assert info["grid"] == 8


@pytest.mark.gpu
@pytest.mark.parametrize("epw", [400000000, INT_MAX])
@pytest.mark.parametrize("d,n,family", [(6, 4, api.FAMILY_REGISTER), (3, 8, api.FAMILY_REGISTER),
                                        (6, 4, api.FAMILY_MATRIX), (3, 4, api.FAMILY_WAVE), (5, 3, api.FAMILY_WAVE),
                                        (2, 8, api.FAMILY_PACKED)])
def test_longest_runs(gpu, d, n, family, epw):
    print(f"[case] d={d} n={n} family={family} epw={epw}", flush=True)
    b = W.random_case(700 + 10 * d + n, d, n, 21, distinct=4)
    db = DeviceBatch(b, device=str(gpu))
    db.run(tuning={"family": family, "entries_per_workgroup": epw})
    err = np.abs(db.output() - oracle.kronmult(b))
    assert float(np.max(err - accumulation_bound(b, np.finfo(np.float64).eps / 2))) <= 0.0
