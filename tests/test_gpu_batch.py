"""Batch functions (source term, Jacobian, E3SM kinetics) across the sizes at
which a launch changes the cells per workgroup: a cell's values are the same
bits in every batch, whole groups or remainders, and a sample equals the
oracle.  Reactant powers and four reactants in a reaction."""
import numpy as np
import pytest

from conftest import golden
from test_lowered import POWERS

pytestmark = pytest.mark.gpu

# around 4, 16 and 64 cells per workgroup and around the sizes a 256-CU card
# switches between them at
SIZES = (1, 3, 5, 255, 2560, 2561, 3072, 3073, 4096, 4097, 10240, 10241, 10300)


def _run_all(torch, fn, inputs, width):
    big = fn(*inputs, torch.full((inputs[0].shape[0], *width), np.nan, dtype=torch.float64, device="cuda"))
    for n in SIZES:
        print("case:", n, "cells", flush=True)
        part = [None if x is None else x[:n].contiguous() for x in inputs]
        out = fn(*part, torch.full((n, *width), np.nan, dtype=torch.float64, device="cuda"))
        assert torch.equal(out, big[:n])
    return big


@pytest.fixture(scope="module")
def cb05(gpu, pkg):
    import importlib
    S = importlib.import_module("tchem-atm_amd.scenarios")
    kmd = pkg.KineticModelData(golden("cb05cl_ae5.yaml"))
    base = pkg.setScenarioConditions(golden("cb05cl_ae5.yaml"), kmd)
    w = S.config1(kmd, base[0], n=max(SIZES))
    return kmd, kmd.createConstData(), gpu.tensor(w.state, device="cuda"), gpu.tensor(w.photo, device="cuda")


def test_source_term_in_every_batch(cb05, gpu, pkg, cb05_oracle):
    kmd, kmcd, state, photo = cb05
    ext = gpu.rand(state.shape[0], kmd.nActive, dtype=gpu.float64, device="cuda")

    def fn(s, p, e, out):
        pkg.SourceTerm.runDeviceBatch(s, p, e, out, kmcd)
        return out

    big = _run_all(gpu, fn, (state, photo, ext), (kmd.nActive,)).cpu().numpy()
    n = 64
    ref = cb05_oracle.sourceterm_batch(state[:n].cpu().numpy(), photo[:n].cpu().numpy()) + ext[:n].cpu().numpy()
    assert np.array_equal(big[:n], ref)


def test_jacobian_in_every_batch(cb05, gpu, pkg, cb05_oracle):
    kmd, kmcd, state, photo = cb05

    def fn(s, p, out):
        pkg.Jacobian.runDeviceBatch(s, p, out, kmcd)
        return out

    big = _run_all(gpu, fn, (state, photo), (kmd.nActive, kmd.nActive))
    n = 16
    ref = cb05_oracle.jacobian_batch(state[:n].cpu().numpy(), photo[:n].cpu().numpy())
    assert np.array_equal(big[:n].cpu().numpy(), ref)
    # an output that is 8-byte aligned only: the same values by 8-byte stores
    m2 = kmd.nActive ** 2
    flat = gpu.zeros(5 * m2 + 1, dtype=gpu.float64, device="cuda")
    pkg.Jacobian.runDeviceBatch(state[:5].contiguous(), photo[:5].contiguous(), flat[1:].view(5, kmd.nActive, -1), kmcd)
    assert gpu.equal(flat[1:].view(5, kmd.nActive, -1), big[:5])


@pytest.mark.parametrize("mode", ["rates", "progress", "net"])
def test_e3sm_kinetics_in_every_batch(mode, gpu, pkg):
    torch = gpu
    kmd = pkg.KineticModelData(golden("uci_v2_test3.yaml"))
    kmcd = kmd.createConstData()
    inp = golden("uci_col_input_conditions.yaml")
    state = pkg.setScenarioConditions(inp, kmd)
    k = state.shape[0]
    rows = np.arange(max(SIZES)) % k
    photo = torch.tensor(pkg.setScenarioConditionsPhotolysisReactions(inp, kmd, k)[rows], device="cuda")
    ext = torch.tensor(pkg.setScenarioConditionsExternalForcing(inp, kmd, k)[rows], device="cuda")
    state = torch.tensor(state[rows], device="cuda")

    def rates(s, out):
        pkg.ReactionRates.runDeviceBatch(s, out, kmcd)
        return out

    def progress(s, p, out):
        pkg.RateofProgress.runDeviceBatch(s, p, out, kmcd)
        return out

    def net(s, p, e, out):
        pkg.NetProductionRates.runDeviceBatch(s, p, e, out, kmcd)
        return out

    if mode == "rates":
        big = _run_all(torch, rates, (state,), (kmd.nReac,))
    elif mode == "progress":
        big = _run_all(torch, progress, (state, photo), (kmd.nReac,))
    else:
        big = _run_all(torch, net, (state, photo, ext), (kmd.nSpec,))
    assert torch.equal(big[:k], big[k:2 * k])  # the column repeats


@pytest.mark.parametrize("four", [False, True])
def test_reactant_powers(four, gpu, pkg, oracle_mod, tmp_path):
    text = POWERS
    if four:
        text = text.replace("    B: 1\n    M: 2\n", "    A: 1\n    B: 1\n    D: 2\n    M: 2\n")
    f = tmp_path / "powers.yaml"
    f.write_text(text)
    kmd = pkg.KineticModelData(str(f))
    kmcd = kmd.createConstData()
    o = oracle_mod.Oracle(str(f))
    state = np.repeat(pkg.setScenarioConditions(str(f), kmd), 7, axis=0)
    state[:, 3:] *= np.random.default_rng(3).uniform(0.5, 2.0, (7, kmd.nSpec))
    d = gpu.tensor(state, device="cuda")
    m = kmd.nActive
    om = gpu.zeros(7, m, dtype=gpu.float64, device="cuda")
    jac = gpu.zeros(7, m, m, dtype=gpu.float64, device="cuda")
    pkg.SourceTerm.runDeviceBatch(d, None, None, om, kmcd)
    pkg.Jacobian.runDeviceBatch(d, None, jac, kmcd)
    np.testing.assert_allclose(om.cpu().numpy(), o.sourceterm_batch(state), rtol=1e-14, atol=0)
    np.testing.assert_allclose(jac.cpu().numpy(), o.jacobian_batch(state), rtol=1e-14, atol=0)
