"""The 16-byte loads of the post-processing kernel (quality_lead, quality_granule_at and quality_granule_skip in
gatk_amd/csrc/pairhmm_kernels.hpp), compiled for the CPU: none begins before the plane or ends after its read, and
together they give every byte of the read once and in order."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PROGRAM = r"""
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <initializer_list>
#include "ROOT/gatk_amd/csrc/pairhmm_kernels.hpp"
using namespace gatk_pairhmm;
int main() {
    const uint64_t plane = 4096 + 5;  // the plane's first byte
    for (int off : {0, 3, 10, 11, 12, 26, 27, 28, 31})
        for (int len = 0; len <= 1100; ++len) {
            const int lead = quality_lead(plane + static_cast<uint64_t>(off), len, plane), span = lead + len;
            int next = 0, k = 0;  // the byte due
            for (; 16 * k < span; ++k) {
                const int at = quality_granule_at(span, k), skip = quality_granule_skip(span, lead, k);
                if (span >= 16 && (at + off - lead < 0 || at + 16 > span))
                    return std::printf("%d %d: load at %d\n", len, k, at), 1;
                for (int b = skip > 0 ? skip : 0; b < 16; ++b)
                    if (at - lead + b != next++) return std::printf("%d %d: byte %d\n", len, k, at - lead + b), 1;
            }
            if (next != len) return std::printf("%d: %d bytes\n", len, next), 1;
            for (; k < 80; ++k)
                if (quality_granule_skip(span, lead, k) < 16) return std::printf("%d %d: past the end\n", len, k), 1;
        }
    return quality_granule_skip(0, 0, 0) < 16;
}
"""


def test_loads_stay_inside_the_plane_and_cover_the_read(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    src, exe = os.path.join(str(tmp_path), "granules.cpp"), os.path.join(str(tmp_path), "granules")
    with open(src, "w") as f:
        f.write(PROGRAM.replace("ROOT", os.path.dirname(HERE)))
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(HERE, "stream_harness"), "-o", exe, src], check=True)
    p = subprocess.run([exe], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout
