"""Every number of cells per workgroup that the cell regions leave room for is
accepted and gives the bits of one cell per workgroup."""
import dataclasses
import importlib

import numpy as np
import pytest

from conftest import golden

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mech,precision,cells", [("carbonbond05.yaml", "fp64", 11),
                                                  ("cb05_soa_gas.yaml", "mixed", 16)])
def test_full_workgroups(gpu, pkg, mech, precision, cells):
    S = importlib.import_module("tchem-atm_amd.scenarios")
    D = importlib.import_module("tchem-atm_amd.driver")
    kmd = pkg.KineticModelData(golden(mech))
    kmcd = kmd.createConstData()
    base = pkg.setScenarioConditions(golden(mech), kmd)[0]
    w = dataclasses.replace(S.config1(kmd, base, n=3 * cells + 2), tend=1e-6)
    form = dict(precision=pkg.PRECISION_MIXED if precision == "mixed" else pkg.PRECISION_FP64, lu=pkg.LU_SPARSE)

    def run(c):
        print("case:", mech, precision, c, "cells", flush=True)
        r = D.DeviceRun(kmcd, w)
        r.reset()
        r.run_to_end(**form, cells_per_block=c)
        gpu.cuda.synchronize()
        return r.state.cpu().numpy()

    single = run(1)
    assert np.all(np.isfinite(single))
    assert np.array_equal(run(cells), single)
