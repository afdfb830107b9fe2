"""Cells whose temperature is NaN or zero: source term and Jacobian give NaN
where the oracle does, also for rate constants without temperature
dependence, and their neighbours in the batch keep their values."""
import numpy as np
import pytest

from conftest import golden

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mech", ["photolysis.yaml", "cb05cl_ae5.yaml"])
@pytest.mark.parametrize("cells", [6, 5000, 12000])  # 4, 16 and 64 cells per workgroup
def test_nan_where_the_oracle_has_nan(gpu, pkg, mech, cells):
    import oracle

    kmd = pkg.KineticModelData(golden(mech))
    kmcd = kmd.createConstData()
    state = np.repeat(pkg.setScenarioConditions(golden(mech), kmd)[:1], cells, axis=0)
    state[1, 2], state[3, 2], state[4, 2] = np.nan, 0.0, np.inf
    photo = np.full((cells, max(kmd.nPhoto, 1)), 1e-4)
    o = oracle.Oracle(golden(mech))
    m = kmd.nActive
    s, p = (gpu.tensor(x, device="cuda") for x in (state, photo))
    p = p if kmd.nPhoto else None
    omega = gpu.zeros(cells, m, dtype=gpu.float64, device="cuda")
    jac = gpu.zeros(cells, m, m, dtype=gpu.float64, device="cuda")
    print("case:", mech, cells, "cells", flush=True)
    pkg.SourceTerm.runDeviceBatch(s, p, None, omega, kmcd)
    pkg.Jacobian.runDeviceBatch(s, p, jac, kmcd)
    ref = o.sourceterm_batch(state[:6], photo[:6])
    assert np.isnan(ref[1]).any() and np.isnan(ref[3]).any()
    assert np.array_equal(omega[:6].cpu().numpy(), ref, equal_nan=True)
    jref = o.jacobian_batch(state[:6], photo[:6])
    assert np.array_equal(np.isnan(jac[:6].cpu().numpy()), np.isnan(jref))
    assert bool((omega[5:] == omega[5]).all()) and bool((jac[5:] == jac[5]).all())
