"""The MFMA form's instances of 4, 6 and 8 tiles per side, at the orders where
the choice changes (127 | 128 and 191 | 192 unknowns) and at the ends of the
range: the batched dense solve against numpy's FP64 solve, and the integrator
on uniformly coupled synthetic mechanisms of 4- and 6-tile size against the
mixed sparse form, which factors the same FP32 matrix.  Tolerances: FP32
factors of these diagonally dominant systems give about 1e-6, a misplaced tile
or right-hand side O(1); the integrator's bar is the mixed form's 1e-4 above
1e-8 ppm.
"""
import ctypes
import dataclasses
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 31, 64, 127, 128, 160, 191, 192, 254])
def test_dense_solve_tile_counts(pkg, gpu, n):
    print("case: dense MFMA solve n =", n, flush=True)
    torch = gpu
    lib = pkg.lib()
    batch = 5
    g = np.random.Generator(np.random.Philox(key=n))
    A = g.uniform(-1.0, 1.0, (batch, n, n)) / np.sqrt(n)
    A[:, np.arange(n), np.arange(n)] += 2.0 + g.uniform(0.0, 1.0, (batch, n))
    b = g.uniform(-1.0, 1.0, (batch, n))
    dA, db = (torch.tensor(v, dtype=torch.float64, device="cuda") for v in (A, b))
    dx = torch.full((batch, n), -7.0, dtype=torch.float64, device="cuda")
    rc = lib.tchem_dense_lu_solve_mfma(n, batch, ctypes.c_void_p(dA.data_ptr()), ctypes.c_void_p(db.data_ptr()),
                                       ctypes.c_void_p(dx.data_ptr()), ctypes.c_void_p(pkg._stream_ptr(None)))
    assert rc == 0, lib.tchem_last_error().decode()
    torch.cuda.synchronize()
    ref = np.linalg.solve(A, b[..., None])[..., 0]
    assert np.abs(dx.cpu().numpy() - ref).max() / np.abs(ref).max() < 2e-5


@pytest.mark.parametrize("species", [40, 130])
def test_integrator_tile_counts(pkg, gpu, tmp_path, species):
    print("case: MFMA integrator,", species, "species", flush=True)
    S = importlib.import_module("tchem-atm_amd.scenarios")
    D = importlib.import_module("tchem-atm_amd.driver")
    mech = S.synthetic_mechanism_yaml(str(tmp_path / "uniform.yaml"), n_species=species, n_reactions=3 * species,
                                      coupling="uniform")
    kmd = pkg.KineticModelData(mech)
    kmcd = kmd.createConstData()
    w, _ = S.config4(kmd, pkg.setScenarioConditions(mech, kmd)[0], size_scale=1 / 64)
    w = dataclasses.replace(w, state=w.state[:6].copy(), photo=w.photo[:6].copy(), tend=3600.0)
    out = {}
    for lu in (pkg.LU_MFMA, pkg.LU_SPARSE):
        run = D.DeviceRun(kmcd, w)
        run.reset()
        run.run_to_end(precision=pkg.PRECISION_MIXED, schedule=pkg.SCHEDULE_PERSISTENT, collect_stats=True, lu=lu)
        gpu.cuda.synchronize()
        out[lu] = (run.state.cpu().numpy()[:, 3:3 + kmd.nActive], run.total_stats.copy())
    (a, sa), (b, sb) = out[pkg.LU_MFMA], out[pkg.LU_SPARSE]
    assert np.all(np.abs(sa[:, 0] - sb[:, 0]) <= 0.02 * sb[:, 0] + 2)
    assert (np.abs(a - b) / np.maximum(np.abs(b), 1e-8)).max() < 1e-4
