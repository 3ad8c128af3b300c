"""The step loops' LDS stores leave the compiler in step order (gatk_amd/csrc/check_isa.py).

Every lane stores its cell at its own column, so a column is stored by all lanes, a step apart, and the last
lane's store has to come last.  The compiler sees one lane, whose addresses differ, and its post-RA
scheduler swaps steps wherever the source does not hold them apart, so the forward kernels are compiled with
it on here, whatever flags the library is built with.
"""
import importlib.util
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "gatk_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"


def _guard():
    path = os.path.join(CSRC, "check_isa.py")
    if not os.path.exists(path):
        pytest.skip("check_isa.py is not present here")
    spec = importlib.util.spec_from_file_location("check_isa", path)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def _asm(*lines):
    return "kernel:\n" + "".join(l + "\n" if l.endswith(":") else f"\t{l}\n" for l in lines)


@pytest.mark.parametrize("lines", [
    ("ds_write_b128 v4, v[0:3] offset:640", "ds_write_b128 v4, v[8:11] offset:672", "ds_write_b128 v4, v[4:7] offset:656"),
    ("ds_write2_b32 v9, v0, v1 offset0:4 offset1:5", "ds_write2_b32 v9, v2, v3 offset0:2 offset1:3"),
    ("ds_write_b64 v9, v[0:1] offset:8", "v_add_f32_e32 v3, v9, v2", "ds_write_b64 v9, v[2:3]"),
])
def test_swapped_steps_are_found(lines):
    assert len(_guard().lds_stores_out_of_order(_asm(*lines))) >= 1


@pytest.mark.parametrize("lines", [
    ("ds_write_b128 v4, v[0:3] offset:640", "ds_write_b128 v4, v[4:7] offset:656", "ds_write_b32 v5, v0 offset:4"),
    ("ds_write_b32 v4, v0 offset:4000", "ds_write_b32 v4, v1 offset:64"),                    # another plane
    ("ds_write_b32 v4, v0 offset:8", "v_add_u32_e32 v4, 32, v4", "ds_write_b32 v4, v0"),     # the next block's columns
    ("ds_write_b32 v4, v0 offset:8", ".LBB0_1:", "ds_write_b32 v4, v0"),
])
def test_ordered_stores_are_not(lines):
    assert _guard().lds_stores_out_of_order(_asm(*lines)) == []


@pytest.mark.parametrize("name", ["pairhmm_fwd.hip", "pdhmm.hip", "sw.hip"])
def test_step_stores_stay_in_order_with_the_post_ra_scheduler(name, tmp_path):
    if not shutil.which(HIPCC):
        pytest.skip("hipcc is not available")
    g = _guard()
    out = str(tmp_path / "kernels.s")
    subprocess.run([HIPCC, *g.FLAGS, "-o", out, os.path.join(CSRC, name)], check=True, stderr=subprocess.DEVNULL)
    with open(out) as f:
        assert g.lds_stores_out_of_order(f.read()) == []
