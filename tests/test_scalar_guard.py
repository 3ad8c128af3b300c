"""The build guard's list of scalar instructions that leave memory as it is (gatk_amd/csrc/check_isa.py), on
hand-written assembly text: whatever is not on it fails the build."""
import importlib.util
import os

import pytest

GUARD = os.path.join(os.path.dirname(__file__), "..", "gatk_amd", "csrc", "check_isa.py")


def _unknown(*lines):
    if not os.path.exists(GUARD):
        pytest.skip("check_isa.py is not present here")
    spec = importlib.util.spec_from_file_location("check_isa", GUARD)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod.unknown_scalar_ops("".join(f"\t{l}\n" for l in lines))


def test_loads_arithmetic_and_control_pass():
    assert _unknown("s_load_dwordx4 s[0:3], s[4:5], 0x10", "s_buffer_load_dword s0, s[4:7], 0", "s_mov_b64 exec, -1",
                    "s_and_saveexec_b64 s[2:3], vcc", "s_cmp_lg_u32 s0, 0", "s_cbranch_scc1 .LBB0_1", "s_branch .LBB0_2",
                    "s_waitcnt vmcnt(0)", "s_nop 4", "s_endpgm", "; s_other_dword in a comment",
                    "ds_write_b32 v0, v1", "global_store_dword v0, v1, s[0:1]") == []


@pytest.mark.parametrize("op", ["s_other_dword", "s_other_dwordx4", "s_buffer_other_dword", "s_other_add", "s_other_swap_x2",
                                "s_other_wb", "s_load_dword_other"])
def test_other_scalar_instructions_are_named(op):
    assert _unknown("s_mov_b32 s0, 0", f"{op} s0, s[2:3], 0x0", "s_endpgm") == [op]
