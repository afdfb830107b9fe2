"""Cells per workgroup chosen from the batch size: around one, two and a full
workgroup of cells per CU of a 256-CU card, and around one and two such waves,
the integrator's results are the bits of one cell per workgroup."""
import dataclasses
import importlib

import numpy as np
import pytest

from conftest import golden

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("schedule", ["grid", "persistent"])
def test_any_batch_has_the_bits_of_single_cells(gpu, pkg, precision, schedule):
    S = importlib.import_module("tchem-atm_amd.scenarios")
    D = importlib.import_module("tchem-atm_amd.driver")
    kmd = pkg.KineticModelData(golden("cb05cl_ae5.yaml"))
    kmcd = kmd.createConstData()
    base = pkg.setScenarioConditions(golden("cb05cl_ae5.yaml"), kmd)[0]
    w = dataclasses.replace(S.config1(kmd, base, n=5700), tend=1e-3)
    form = dict(precision=pkg.PRECISION_MIXED if precision == "mixed" else pkg.PRECISION_FP64,
                schedule=pkg.SCHEDULE_GRID if schedule == "grid" else pkg.SCHEDULE_PERSISTENT, lu=pkg.LU_SPARSE)

    def run(n, **more):
        r = D.DeviceRun(kmcd, dataclasses.replace(w, state=w.state[:n].copy(), photo=w.photo[:n].copy()))
        r.reset()
        r.run_to_end(**form, **more)
        gpu.cuda.synchronize()
        return r.state.cpu().numpy()

    single = run(w.n, cells_per_block=1)
    assert np.all(np.isfinite(single))
    for n in (1, 255, 257, 513, 2816, 2817, 4097, 5633, 5700):
        print("case:", n, "cells", precision, schedule, flush=True)
        assert np.array_equal(run(n), single[:n])
