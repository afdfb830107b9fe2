"""The device encoding of the compiled programs (tchem-atm_amd/csrc/lowered.cpp),
run on the CPU by tests/native/lowered_check.cpp against the rounds it was
lowered from: every value bit for bit (zeros may differ in sign), FP32 and
FP64, forward, transposed and aerosol programs, no access outside the cell
region or the stream."""
import os
import subprocess

import pytest

from conftest import ROOT, golden

CSRC = os.path.join(ROOT, "tchem-atm_amd", "csrc")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("native") / "lowered_check")
    srcs = [os.path.join(ROOT, "tests", "native", "lowered_check.cpp")] + [
        os.path.join(CSRC, f) for f in ("yaml_lite.cpp", "kinetic_model.cpp", "mechanism.cpp", "schedule.cpp",
                                        "aerosol_model.cpp", "lowered.cpp")]
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + CSRC, *srcs, "-o", exe], check=True)
    return exe


def _run(*args):
    r = subprocess.run(args, capture_output=True, text=True)
    print(r.stdout[-2000:])
    assert r.returncode == 0, r.stdout[-3000:]
    return r.stdout


# one reaction, sources only, powers of reactants, the largest shipped
# mechanism, and the E3SM one (64 > species)
@pytest.mark.parametrize("mech", ["troe.yaml", "emission.yaml", "cb05cl_ae5.yaml", "uci_v2_test3.yaml"])
def test_encoded_programs_equal_the_rounds(checker, mech):
    _run(checker, golden(mech))


def test_encoded_aerosol_programs_equal_the_rounds(checker):
    _run(checker, golden("cb05_soa_gas.yaml"), golden("cb05_soa_aero.yaml"))


# more than 128 unknowns and cell regions above 64 KiB: shifted address
# fields, several masks per section, unfused multiplier rounds
@pytest.mark.parametrize("n_species,n_reactions", [(129, 200), (180, 400)])
def test_encoded_programs_with_shifted_fields(checker, pkg, tmp_path, n_species, n_reactions):
    import importlib
    S = importlib.import_module("tchem-atm_amd.scenarios")
    f = S.synthetic_mechanism_yaml(str(tmp_path / "m.yaml"), seed=5, n_species=n_species, n_reactions=n_reactions,
                                   n_radicals=8, window=20, coupling="cascade")
    out = _run(checker, f)
    assert "shift 2" in out and "shift 3" in out
