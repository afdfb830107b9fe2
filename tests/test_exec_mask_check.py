"""The build's check of its device code (tchem-atm_amd/csrc/check_exec_mask.py):
vector registers stored before a join restores the lane mask are refused,
the ordinary forms of a join are not, and the library's Makefile runs it."""
import importlib.util
import os
import subprocess
import sys

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "tchem-atm_amd", "csrc")
SCRIPT = os.path.join(CSRC, "check_exec_mask.py")


@pytest.fixture(scope="module")
def check():
    spec = importlib.util.spec_from_file_location("check_exec_mask", SCRIPT)
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


HEAD = """kernel_of_a_join:
	s_mov_b64 s[2:3], exec
	s_and_b64 s[4:5], s[2:3], s[4:5]
	s_mov_b64 exec, s[4:5]
	s_cbranch_execz .LBB0_2
; %bb.1:
	global_load_dwordx2 v[74:75], v[2:3], off
.LBB0_2:
"""
TAIL = """	s_add_i32 s2, s70, 8
	scratch_load_dwordx2 v[2:3], off, off offset:116 ; 8-byte Folded Reload
	s_endpgm
"""
RESTORE = "	s_or_b64 exec, exec, s[2:3]\n"
SPILL = "	scratch_store_dwordx2 off, v[10:11], off offset:116 ; 8-byte Folded Spill\n"


# the join of the 4-slot aerosol integrator as it was compiled with spills
@pytest.mark.parametrize("early", [
    "	v_writelane_b32 v254, s6, 9\n	s_waitcnt vmcnt(2)\n" + SPILL,
    "	v_accvgpr_write_b32 a3, v10\n",
    "	v_mov_b32_e32 v40, v10\n",
])
def test_stores_before_the_mask_is_restored_are_found(check, early):
    found = check.find((HEAD + early + RESTORE + TAIL).splitlines())
    assert [(f[0], f[1]) for f in found] == [("kernel_of_a_join", ".LBB0_2")]


def test_a_spill_before_the_restore_of_a_join_without_a_branch_is_found(check):
    text = HEAD.replace("	s_cbranch_execz .LBB0_2\n", "").replace(".LBB0_2:", "; %bb.2:") + SPILL + RESTORE + TAIL
    assert [f[1] for f in check.find(text.splitlines())] == ["%bb.2"]


@pytest.mark.parametrize("early", ["", "	v_writelane_b32 v254, s6, 9\n	v_readlane_b32 s7, v252, 17\n"])
def test_joins_that_restore_the_mask_first_pass(check, early):
    assert check.find((HEAD + early + RESTORE + SPILL + TAIL).splitlines()) == []


def test_the_status_tells(tmp_path):
    for name, text, rc in (("bad.s", HEAD + SPILL + RESTORE + TAIL, 1), ("good.s", HEAD + RESTORE + SPILL + TAIL, 0)):
        f = tmp_path / name
        f.write_text(text)
        assert subprocess.run([sys.executable, SCRIPT, str(f)], capture_output=True).returncode == rc


def test_spilling_kernels_are_named(check):
    meta = "    .name:           _Z1aPf\n    .sgpr_spill_count: 9\n    .vgpr_spill_count: %d\n"
    assert check.spills((meta % 0).splitlines()) == {}
    assert check.spills((meta % 155 + (meta % 0).replace("1a", "1b")).splitlines()) == {"_Z1aPf": 155}


def test_the_library_is_built_through_the_check():
    """make would check the assembly of the compilation whose object it links."""
    r = subprocess.run(["make", "-n", "-B", "-C", CSRC, "_build/kernels.o"], capture_output=True, text=True, check=True)
    lines = [ln for ln in r.stdout.splitlines() if "kernels" in ln]
    compiled = next(i for i, ln in enumerate(lines) if "-save-temps=obj" in ln and "kernels.hip" in ln)
    checked = next(i for i, ln in enumerate(lines) if "check_exec_mask.py" in ln and "gfx950.s" in ln)
    kept = next(i for i, ln in enumerate(lines) if ln.startswith("mv "))
    assert compiled < checked < kept
