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


def test_encoded_programs_of_reactant_powers(checker, tmp_path):
    """Powers 0 (a fractional coefficient), 1, 2, 3 and 4, one of them on a
    constant species; every derivative factor of each."""
    f = tmp_path / "powers.yaml"
    f.write_text(POWERS)
    _run(checker, str(f))


POWERS = """NCAR-version: v1.0
environmental_conditions:
  pressure:
    initial_value: [101325]
    units: Pa
  temperature:
    initial_value: [298.0]
    units: K
initial_state:
  A:
    initial_value: [0.1]
    units: mol m-3
  B:
    initial_value: [0.2]
    units: mol m-3
  D:
    initial_value: [0.3]
    units: mol m-3
  M:
    initial_value: [10.0]
    units: mol m-3
constant_species:
- description: third body
  name: M
species:
- description: a
  name: A
- description: b
  name: B
- description: d
  name: D
reactions:
- MUSICA_name: R1
  reactants:
    A: 3
    B: 2
    M: 1
  products:
    D: 1
  type: ARRHENIUS
  coefficients:
    A: 2.0
- MUSICA_name: R2
  reactants:
    A: 0.5
    D: 4
  products:
    B: 2
  type: ARRHENIUS
  coefficients:
    A: 0.5
    C: -10.0
- MUSICA_name: R3
  reactants:
    B: 1
    M: 2
  products:
    A: 1
  type: ARRHENIUS
  coefficients:
    A: 1.5
    B: 0.3
"""
