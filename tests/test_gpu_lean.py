"""The lean kernels (plain sites of a box with a geometry map: scalar plane and
row offsets, flat even steps, pairs) with the launch over the rows that hold
other codes, against the general kernel over every row: one step from the same
state, each storage form and pattern, at row lengths below, between and on
whole waves and blocks, walls as whole rows and inside rows, with a force
field, overlaps, and the passive scalar.  Tolerance as for the row lists: 16
epsilons of an array's scale, one for stored 2-byte values."""
import numpy as np
import pytest
import torch

from pytnl_lbm import ADE_GEO, D3Q7Lattice, _abi
from pytnl_lbm._abi import GEO
from test_gpu_row_lists import fields, lattice, units, within

pytestmark = pytest.mark.gpu

FORMS = ["f64", "f32", "f32dev", "f16dev", "bf16dev", "i16dev"]


def geometry(kind, X, Y, Z):
    """"walls": z walls, everything else periodic.  "duct": walls on the y and z
    faces, fluid inside.  "few": the duct with one inlet row and one symmetry
    site, so that a few rows hold other codes."""
    geo = np.full((X, Y, Z), GEO.PERIODIC if kind == "walls" else GEO.FLUID, dtype=np.int16)
    geo[:, :, 0] = geo[:, :, -1] = GEO.WALL
    if kind != "walls":
        geo[:, 0, :] = geo[:, -1, :] = GEO.WALL
    if kind == "few":
        geo[1, 1:-1, 2] = GEO.INFLOW
        geo[2, Y // 2, 3] = GEO.SYM_TOP
    return geo


def both(X, Y, Z, storage, pattern, geo, **kw):
    a, b = (lattice(X, Y, Z, storage, pattern, geo, rl, **kw) for rl in (True, False))
    assert a.d.row_count[0] * 8 <= X * Z and not b.d.rows
    return a, b


@pytest.mark.parametrize("kind", ["walls", "duct", "few"])
@pytest.mark.parametrize("shape", [(4, 7, 6), (3, 64, 8), (4, 70, 6), (4, 97, 5), (3, 128, 7), (3, 257, 6), (2, 512, 9)])
@pytest.mark.parametrize("pattern", ["AA", "AB"])
@pytest.mark.parametrize("storage", FORMS)
def test_lean_step_matches_general_kernel(storage, pattern, shape, kind):
    X, Y, Z = shape
    if kind == "few" and X < 3:
        X = 3
    a, b = both(X, Y, Z, storage, pattern, geometry(kind, X, Y, Z), force=(1e-5, 0.0, -2e-6))
    for lat in (a, b):
        lat.set_inflow(0.02, 0.0, 0.01)
        lat.set_equilibrium_field(*fields(X, Y, Z, 3))
    for t in range(4):
        for x, y in zip(a.df, b.df):
            x.copy_(y)
        a.step(output_macro=t > 1)
        b.step(output_macro=t > 1)
        torch.cuda.synchronize()
        for x, y in zip(a.df + [a.macro], b.df + [b.macro]):
            assert within(x, y), (storage, pattern, shape, kind, t, units(x, y))


@pytest.mark.parametrize("pattern", ["AA", "AB"])
@pytest.mark.parametrize("storage,shape", [("f64", (80, 256, 64)), ("f16dev", (200, 256, 96))])
def test_lean_step_beyond_the_cache(storage, shape, pattern):
    """Arrays above the last-level cache in whole rows: the row form with hints."""
    X, Y, Z = shape
    a, b = both(X, Y, Z, storage, pattern, geometry("few", X, Y, Z))
    for lat in (a, b):
        lat.set_inflow(0.02, 0.0, 0.01)
        lat.set_equilibrium_field(*fields(X, Y, Z, 3))
    for t in range(2):
        for x, y in zip(a.df, b.df):
            x.copy_(y)
        a.step()
        b.step()
        torch.cuda.synchronize()
        for x, y in zip(a.df, b.df):
            assert within(x, y), (storage, pattern, t, units(x, y))


@pytest.mark.parametrize("pattern", ["AA", "AB"])
@pytest.mark.parametrize("flags", [0, _abi.FLAG_DISTRIBUTED_X])
def test_overlaps_and_force_field(pattern, flags):
    """Overlaps on an axis that is not distributed: the wrap and the clamp of the
    two kinds of sites differ at the faces."""
    X, Y, Z = 5, 70, 6
    geo = geometry("few", X, Y, Z)
    a, b = both(X, Y, Z, "f64", pattern, geo, overlap=(1, 1, 1))
    rng = np.random.default_rng(2)
    force = [1e-5 * rng.standard_normal((X + 2, Y + 2, Z + 2)) for _ in range(3)]
    start = torch.as_tensor(rng.random(a.df[0].numel()) * 0.01 + 0.03)
    for lat in (a, b):
        lat.set_force_field(*force)
    for t in range(3):
        for lat in (a, b):
            for d in lat.df:
                d.copy_(start)
            lat.step(output_macro=True, flags=flags)
        torch.cuda.synchronize()
        for x, y in zip(a.df + [a.macro], b.df + [b.macro]):
            assert within(x, y), (pattern, flags, t, units(x, y))


@pytest.mark.parametrize("kind", ["walls", "duct", "few"])
@pytest.mark.parametrize("Y", [33, 64, 100, 256])
@pytest.mark.parametrize("pattern", ["AA", "AB"])
@pytest.mark.parametrize("storage", ["f64", "f32", "f16dev", "i16dev"])
def test_coupled_lean_step_matches_general_kernel(storage, pattern, Y, kind):
    X, Z = 4, 6
    geo = geometry(kind, X, Y, Z)
    ageo = np.full((X, Y, Z), ADE_GEO.PERIODIC if kind == "walls" else ADE_GEO.FLUID, dtype=np.int16)
    ageo[:, :, 0] = ageo[:, :, -1] = ADE_GEO.WALL
    if kind == "few":
        ageo[1, 1:-1, 2] = ADE_GEO.INFLOW
    src = np.random.default_rng(7).standard_normal((X, Y, Z)) * 1e-3
    pair = []
    for nse in both(X, Y, Z, storage, pattern, geo):
        ade = D3Q7Lattice(nse, collision="CLBM", diffusivity=0.02, geo=ageo, phi_ref=0.1, store_scale=50.0)
        nse.set_equilibrium_field(*fields(X, Y, Z, 5))
        ade.set_equilibrium(0.1)
        ade.set_source(src)
        ade.set_inflow(0.15)
        pair.append((nse, ade))
    (na, aa), (nb, ab) = pair
    for t in range(4):
        for x, y in zip(na.df + aa.df, nb.df + ab.df):
            x.copy_(y)
        na.step_coupled(aa, output_macro=True)
        nb.step_coupled(ab, output_macro=True)
        torch.cuda.synchronize()
        for x, y in zip(na.df + aa.df + [na.macro, aa.phi], nb.df + ab.df + [nb.macro, ab.phi]):
            assert within(x, y), (storage, pattern, Y, kind, t, units(x, y))
