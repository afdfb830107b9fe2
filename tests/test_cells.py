"""Cells of the sparse forms that fit a workgroup (tests/native/cells_check.cpp):
at least as many as the items of a cell (factor entries, right-hand side and
pivots, derivative pairs, concentrations, rate constants, rates of progress,
segment sums) leave room for, with or without staged tolerances, so that no number of cells per workgroup that
such a cell allows is refused or given up.  And the regions that share room
for it, over several iterations on one cell (lowered_repeat_check.cpp)."""
import importlib
import os
import random
import re
import subprocess

import pytest

from conftest import ROOT, golden

CSRC = os.path.join(ROOT, "tchem-atm_amd", "csrc")


def _build(tmp_path_factory, name):
    exe = str(tmp_path_factory.mktemp("native") / name)
    srcs = [os.path.join(ROOT, "tests", "native", name + ".cpp")] + [
        os.path.join(CSRC, f) for f in ("yaml_lite.cpp", "kinetic_model.cpp", "mechanism.cpp", "schedule.cpp",
                                        "aerosol_model.cpp", "lowered.cpp")]
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC, *srcs,
                    "-o", exe], check=True)
    return exe


@pytest.fixture(scope="module")
def cells(tmp_path_factory):
    exe = _build(tmp_path_factory, "cells_check")

    def run(*args):
        out = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, check=True).stdout
        return [[int(x) for x in re.findall(r"\d+", ln)] for ln in out.splitlines()]
    return run


@pytest.fixture(scope="module")
def repeat(tmp_path_factory):
    return _build(tmp_path_factory, "lowered_repeat_check")


# (FP64 in memory, staged), (FP32 in memory, staged)
@pytest.mark.parametrize("mech,fp64,fp32", [
    ("cb05cl_ae5.yaml", (11, 6), (16, 10)),
    ("carbonbond05.yaml", (11, 6), (16, 9)),
    ("cb05_soa_gas.yaml", (10, 6), (16, 9)),
    ("uci_v2_test3.yaml", (12, 12), (16, 16)),
    ("troe.yaml", (12, 12), (16, 16)),
    ("cascade129", (7, 3), (8, 5)),
    ("cascade180", (3, 0), (6, 0)),
    ("uniform60", (6, 0), (10, 0)),
])
def test_gas_cells_per_workgroup(cells, pkg, tmp_path, mech, fp64, fp32):
    S = importlib.import_module("tchem-atm_amd.scenarios")
    f = golden(mech) if mech.endswith(".yaml") else str(tmp_path / "m.yaml")
    if mech == "cascade129":
        S.synthetic_mechanism_yaml(f, seed=5, n_species=129, n_reactions=200, n_radicals=8, window=20, coupling="cascade")
    elif mech == "cascade180":
        S.synthetic_mechanism_yaml(f, seed=5, n_species=180, n_reactions=400, n_radicals=8, window=20, coupling="cascade")
    elif mech == "uniform60":
        S.synthetic_mechanism_yaml(f, n_species=60, n_reactions=180)
    (_, *d), (_, *s) = cells(f)
    print(mech, "FP64", d, "FP32", s)
    assert all(x >= y for x, y in zip(d, fp64)) and all(x >= y for x, y in zip(s, fp32))


def test_aerosol_cells_per_workgroup(cells):
    want = {1: 8, 5: 8, 8: 7, 20: 5, 30: 4, 35: 3}
    got = {n: c for n, c in cells(golden("cb05_soa_gas.yaml"), golden("cb05_soa_aero.yaml"), *want)}
    print(got)
    assert all(got[n] >= want[n] for n in want)


# few reactions and no pairs, an idle half wavefront, partial sums, shifted
# fields; the aerosol ones with more than 128 unknowns too
@pytest.mark.parametrize("mech", ["emission.yaml", "troe.yaml", "cb05cl_ae5.yaml", "carbonbond05.yaml",
                                  "uci_v2_test3.yaml", "cascade129", "uniform30"])
def test_iterations_on_one_cell(repeat, pkg, tmp_path, mech):
    S = importlib.import_module("tchem-atm_amd.scenarios")
    f = golden(mech) if mech.endswith(".yaml") else str(tmp_path / "m.yaml")
    if mech == "cascade129":
        S.synthetic_mechanism_yaml(f, seed=5, n_species=129, n_reactions=200, n_radicals=8, window=20, coupling="cascade")
    elif mech == "uniform30":
        S.synthetic_mechanism_yaml(f, n_species=30, n_reactions=300)
    r = subprocess.run([repeat, f], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-2000:]


@pytest.mark.parametrize("particles", [1, 5, 20, 24])
def test_iterations_on_one_aerosol_cell(repeat, particles):
    r = subprocess.run([repeat, golden("cb05_soa_gas.yaml"), golden("cb05_soa_aero.yaml"), str(particles)],
                       capture_output=True, text=True)
    print(r.stdout[-1500:])
    assert r.returncode == 0, r.stdout[-2000:]


def test_many_distinct_coefficients(repeat, pkg, tmp_path):
    """8500 yields, all different, in a small cell: more than 16 bits of byte
    address for the coefficient table."""
    species = ["S%02d" % i for i in range(64)]
    rng = random.Random(1)
    out = ["NCAR-version: v1.0", "environmental_conditions:", "  pressure:", "    initial_value: [101325]", "    units: Pa", "  temperature:",
           "    initial_value: [298.0]", "    units: K", "initial_state:"]
    for s in species + ["M"]:
        out += [f"  {s}:", "    initial_value: [0.1]", "    units: mol m-3"]
    out += ["constant_species:", "- description: third body", "  name: M", "species:"]
    out += [ln for s in species for ln in (f"- description: {s}", f"  name: {s}")] + ["reactions:"]
    for r in range(170):
        names = rng.sample(species, 51)
        out += [f"- MUSICA_name: R{r + 1}", "  reactants:", f"    {names[0]}: 1", "  products:"]
        out += [f"    {s}: {rng.uniform(0.1, 1.0)!r}" for s in names[1:]]
        out += ["  type: ARRHENIUS", "  coefficients:", "    A: 1.0"]
    f = tmp_path / "m.yaml"
    f.write_text("\n".join(out) + "\n")
    r = subprocess.run([repeat, str(f)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-500:]
