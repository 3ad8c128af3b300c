"""Which packed launches take the split kernel (takes_split in gatk_amd/csrc/pairhmm_kernels.hpp), compiled
for the CPU: the tuning's waves per block and loop body belong to the packed kernel and keep it, and a grid
over the resident one does not widen the range of the rule."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PROGRAM = r"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstdlib>
#include "ROOT/gatk_amd/csrc/pairhmm_kernels.hpp"
using namespace gatk_pairhmm;
int main(int, char **a) {
    LaunchShape s;
    s.waves_per_block = 4;
    s.packed = std::atoi(a[1]) != 0;
    s.tuned = std::atoi(a[2]) != 0;
    s.grid_percent = std::atoi(a[3]);
    std::printf("%d\n", takes_split(s, static_cast<uint32_t>(std::atoll(a[4])), std::atoi(a[5])) ? 1 : 0);
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    d = str(tmp_path_factory.mktemp("rule"))
    src, exe = os.path.join(d, "rule.cpp"), os.path.join(d, "rule")
    with open(src, "w") as f:
        f.write(PROGRAM.replace("ROOT", os.path.dirname(HERE)))
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(HERE, "stream_harness"), "-o", exe, src], check=True)
    return lambda *a: subprocess.run([exe] + [str(x) for x in a], capture_output=True, text=True, check=True).stdout.strip() == "1"


@pytest.mark.parametrize("packed,tuned,percent,n_items,grid,split", [
    (1, 0, 100, 1, 1, True),
    (1, 0, 100, 40959, 1280, True),    # fewer than eight for each of 5,120 waves
    (1, 0, 100, 40960, 1280, False),
    (1, 1, 100, 1024, 256, False),     # waves per block or loop body asked for
    (0, 0, 100, 1024, 256, False),     # aligned stripes
    (1, 0, 200, 40959, 2560, True),    # a larger grid keeps the resident one's range
    (1, 0, 200, 40960, 2560, False),
    (1, 0, 400, 60000, 5120, False),
    (1, 0, 50, 20479, 640, True),      # a smaller one has longer chunks
    (1, 0, 50, 20480, 640, False),
])
def test_rule(rule, packed, tuned, percent, n_items, grid, split):
    assert rule(packed, tuned, percent, n_items, grid) is split
