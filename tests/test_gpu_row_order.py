"""The A-A steps over row lists (deviation forms, coupled) run the rows that hold other codes first: a site whose
code pulls from another site's slots (OUTFLOW_RIGHT of either lattice) reads them as
they were before the step.  Against launches over sub-boxes, which take no lists: the
outlet's plane, then the rest.  Tolerance as for the row lists: 16 epsilons of an
array's scale, one for stored 2-byte values."""
import numpy as np
import pytest
import torch

from pytnl_lbm import ADE_GEO, D3Q7Lattice
from pytnl_lbm._abi import GEO
from test_gpu_row_lists import fields, lattice, units, within

pytestmark = pytest.mark.gpu

# (18, ., 20): a tenth of the rows hold other codes, a tenth are walls (the even step of the 2-byte forms
# takes pairs); (9, ., 12): a fifth hold other codes; (5, ., 8): a third
SPARSE = [(18, 33, 20), (18, 70, 20)]
DENSE = [(9, 70, 12), (5, 70, 8)]


def channel(X, Y, Z, g):
    """Inlet at x = 0, outlet at x = X - 1, z walls, and an inlet site alone in a row of plain ones."""
    geo = np.full((X, Y, Z), g.FLUID, dtype=np.int16)
    geo[:, :, 0] = geo[:, :, -1] = g.WALL
    geo[0, :, 1:-1] = g.INFLOW
    geo[-1, :, 1:-1] = g.OUTFLOW_RIGHT
    geo[1, 7, 4] = g.INFLOW
    return geo


def outlet_first(lat, step):
    t = lat.iterations
    step(offset=(lat.X - 1, 0, 0))
    lat.iterations = t
    step(end=(lat.X - 1, lat.Y, lat.Z))


@pytest.mark.parametrize("shape,storage", [(s, f) for s in SPARSE + DENSE for f in ("f32dev", "f16dev", "bf16dev", "i16dev")])
def test_step(storage, shape):
    X, Y, Z = shape
    geo = channel(X, Y, Z, GEO)
    a, b = (lattice(X, Y, Z, storage, "AA", geo, rl) for rl in (True, False))
    assert (a.d.row_count[0] * 8 <= X * Z) == (shape in SPARSE) and (a.d.row_count[0] * 4 <= X * Z) == (X > 5)
    for lat in (a, b):
        lat.set_inflow(0.02, 0.0, 0.01)
        lat.set_equilibrium_field(*fields(X, Y, Z, 3))
    for t in range(4):
        for x, y in zip(a.df, b.df):
            x.copy_(y)
        a.step(output_macro=True)
        outlet_first(b, lambda **kw: b.step(output_macro=True, **kw))
        torch.cuda.synchronize()
        for x, y in zip(a.df + [a.macro], b.df + [b.macro]):
            assert within(x, y), (storage, shape, t, units(x, y))


@pytest.mark.parametrize("shape,storage", [(s, f) for s in SPARSE + DENSE for f in ("f64", "f32", "f16dev", "i16dev")])
def test_coupled_step(storage, shape):
    X, Y, Z = shape
    pair = []
    for rl in (True, False):
        nse = lattice(X, Y, Z, storage, "AA", channel(X, Y, Z, GEO), rl)
        ade = D3Q7Lattice(nse, collision="CLBM", diffusivity=0.02, geo=channel(X, Y, Z, ADE_GEO), phi_ref=0.1,
                          store_scale=50.0)
        nse.set_inflow(0.02, 0.0, 0.01)
        nse.set_equilibrium_field(*fields(X, Y, Z, 5))
        ade.set_equilibrium(torch.as_tensor(0.1 + 0.01 * np.random.default_rng(6).random((X, Y, Z))))
        ade.set_inflow(0.15)
        pair.append((nse, ade))
    (na, aa), (nb, ab) = pair
    for t in range(4):
        for x, y in zip(na.df + aa.df, nb.df + ab.df):
            x.copy_(y)
        na.step_coupled(aa, output_macro=True)
        outlet_first(nb, lambda **kw: nb.step_coupled(ab, output_macro=True, **kw))
        torch.cuda.synchronize()
        for x, y in zip(na.df + aa.df + [na.macro, aa.phi], nb.df + ab.df + [nb.macro, ab.phi]):
            assert within(x, y), (storage, shape, t, units(x, y))
