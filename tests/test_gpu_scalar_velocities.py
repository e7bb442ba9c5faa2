"""The scalar gradient run whose coupled steps write the last segment's
velocities: the gradient equals, bit for bit, one whose backward pass runs every
segment again, also on a second backward pass over the same graph, and the
lattices' own output fields are left alone."""
import numpy as np
import pytest
import torch

from pytnl_lbm import ADE_GEO, GEO, CoupledScalarRun, D3Q7Lattice, D3Q27Lattice, _abi, scalar_run, top_layer_variance

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,macro", [("f64", None), ("f32", _abi.REAL_F64), ("f16dev", None)])
@pytest.mark.parametrize("T,K,host", [(1, None, False), (7, 3, False), (9, 3, True), (5, 5, False), (6, 1, False)])
def test_kept_velocities_give_the_recomputed_gradient(storage, macro, T, K, host):
    X, Y, Z = 9, 13, 8
    geo = torch.full((X, Y, Z), GEO.PERIODIC, dtype=torch.int16)
    geo[:, :, 0] = geo[:, :, -1] = GEO.WALL
    kw = {} if macro is None else {"macro_real": macro}
    lat = D3Q27Lattice(X, Y, Z, storage=storage, pattern="AB", nu=0.01, geo=geo, **kw)
    rng = np.random.default_rng(T)
    lat.set_equilibrium_field(np.ones((X, Y, Z)), *(0.03 * rng.standard_normal((3, X, Y, Z))))
    ageo = torch.full((X, Y, Z), ADE_GEO.PERIODIC, dtype=torch.int16)
    ageo[:, :, 0] = ageo[:, :, -1] = ADE_GEO.WALL
    ade = D3Q7Lattice(lat, collision="CLBM", diffusivity=0.0125, geo=ageo, store_scale=100.0)
    ade.set_equilibrium(0.0)
    lat.macro.fill_(3)
    ade.phi.fill_(5)
    f0, g0 = lat.df[0].clone(), ade.df[0].clone()
    run = CoupledScalarRun(lat, ade, T, K, host_checkpoints=host)
    q = torch.tensor(1e-3 * rng.random(lat.d.XYZ), device="cuda", requires_grad=True)
    loss = top_layer_variance(scalar_run(run, q, g0, f0), lat, 3)
    grads = [torch.autograd.grad(loss, q, retain_graph=True)[0] for _ in range(2)]
    run.held = None  # as if nothing had been kept
    again = torch.autograd.grad(loss, q)[0]
    assert torch.equal(grads[0], again) and torch.equal(grads[1], again) and float(again.abs().max()) > 0
    with torch.no_grad():
        plain = scalar_run(run, q, g0, f0)
    assert torch.equal(loss.detach(), top_layer_variance(plain, lat, 3))
    assert bool((lat.macro == 3).all()) and bool((ade.phi == 5).all())
