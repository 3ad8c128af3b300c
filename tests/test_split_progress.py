"""The progress words of the split stripes (gatk_amd/csrc/pairhmm_kernels.hpp), compiled for the CPU.

A stripe waits on a word that holds the progress of the stripe before it, or still that of the stripe four
earlier, which has ended, or already that of the stripe four later.  The first and the last let it go on as
soon as the asked steps are done, the earlier one never does: also where the stripe's number passes what
the word holds of it (reads over 262,141 bases).
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PROGRAM = r"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include <initializer_list>
#include "../gatk_amd/csrc/pairhmm_kernels.hpp"
using namespace gatk_pairhmm;
int main() {
    const uint32_t steps[] = {72, 448, 5000};
    for (uint32_t s = 0; s < 40000; ++s)
        for (uint32_t total : steps)
            for (uint32_t need : {1u, 64u, total}) {
                const uint32_t want = split_progress(s, need);
                const bool ok = split_reached(split_progress(s, need), want) && split_reached(split_progress(s, total), want) &&
                                !split_reached(split_progress(s, need - 1), want) && split_reached(split_progress(s + 4, 8), want) &&
                                !(s >= 4 && split_reached(split_progress(s - 4, total), want)) && !(s < 4 && split_reached(0, want));
                if (!ok) {
                    std::printf("stripe %u of %u steps, %u asked\n", s, total, need);
                    return 1;
                }
            }
    return 0;
}
"""


def test_waits_hold_past_the_stripe_number_of_a_word(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    src, exe = os.path.join(str(tmp_path), "progress.cpp"), os.path.join(str(tmp_path), "progress")
    with open(src, "w") as f:
        f.write(PROGRAM.replace('"../gatk_amd/', '"' + os.path.dirname(HERE) + "/gatk_amd/"))
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(HERE, "stream_harness"), "-o", exe, src], check=True)
    p = subprocess.run([exe], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout
