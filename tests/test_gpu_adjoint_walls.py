"""The adjoint step where walls of the y faces hand their contributions to the
site one row in: rows of three sites and up, pairs split between two waves, and
every kind of site one row in (fluid, wall, outlet, nothing), against the oracle's
adjoint of the same step, with the tolerances of the adjoint step's other tests."""
import numpy as np
import pytest
import torch

import oracle as O
from lbm_common import rel_max
from pytnl_lbm import D3Q27Lattice, _abi
from pytnl_lbm._abi import GEO
from test_gpu_adjoint import STORE, TORCH, from_dev, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(5, 3, 6), (4, 4, 5), (4, 21, 13), (3, 65, 66), (5, 128, 4), (3, 63, 9)])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("storage,tol", [("f64", 1e-12), ("f32", 2e-5)])
def test_matches_oracle(shape, mixed, storage, tol):
    X, Y, Z = shape
    rng = np.random.default_rng(Y + Z)
    geo = np.full((X, Y, Z), GEO.FLUID, dtype=np.int16)
    geo[:, 0] = geo[:, -1] = geo[:, :, 0] = geo[:, :, -1] = GEO.WALL
    if mixed:
        geo[rng.random((X, Y, Z)) < 0.15] = GEO.WALL
        geo[rng.random((X, Y, Z)) < 0.1] = GEO.PERIODIC
        geo[rng.random((X, Y, Z)) < 0.05] = GEO.OUTFLOW_EQ
        geo[rng.random((X, Y, Z)) < 0.05] = GEO.NOTHING
    force = (1e-4, -2e-4, 5e-5)
    mreal = _abi.REAL_F64 if storage == "f64" else _abi.REAL_F32
    g = D3Q27Lattice(X, Y, Z, storage=storage, pattern="AB", nu=0.02, geo=geo, force=force, macro_real=mreal)
    h = O.HostLattice(X, Y, Z, storage=STORE[storage], pattern=_abi.PATTERN_AB, nu=0.02, geo=geo, force=force,
                      macro_real=mreal, threads=8)
    r = [1 + 0.01 * rng.standard_normal((X, Y, Z))] + list(0.03 * rng.standard_normal((3, X, Y, Z)))
    h.set_equilibrium_field(*r)
    h.import_f64(h.export_f64(0) * (1 + 0.02 * rng.standard_normal((27, X, Y, Z))), which=0)
    g.import_f64(h.export_f64(0), which=0)
    wq = from_dev(to_dev(rng.standard_normal((27, X, Y, Z)), TORCH[storage]), X, Y, Z)
    ref = h.adjoint_step(wq, grad=np.zeros((3, Z, Y)), which=0)
    lam = torch.empty(27 * g.d.XYZ, dtype=TORCH[storage], device="cuda")
    g.adjoint_step(to_dev(wq, TORCH[storage]), lam, torch.zeros(3 * Y * Z, dtype=torch.float64, device="cuda"), which=0)
    torch.cuda.synchronize()
    got = from_dev(lam, X, Y, Z)
    assert rel_max(got, ref) < tol, rel_max(got, ref)
