"""tnl_lbm_set_wide_addressing chooses between the addressings of one kernel, never
between kernels: the same bits under both settings where the step takes row lists
(the lean kernels and the launch over the rows with other codes), where the periodic
odd step walks the plane, and in every form of the adjoint step."""
import ctypes as C

import numpy as np
import pytest
import torch

from pytnl_lbm import ADE_GEO, D3Q7Lattice, D3Q27Lattice
from pytnl_lbm.adjoint import tape_elements
from pytnl_lbm.lattice import _ptr, _stream_ptr
from test_gpu_addressing import bits, both_ways, duct, fields
from test_gpu_row_lists import lattice

pytestmark = pytest.mark.gpu

# a tenth of the rows hold the duct's inlet and outlet codes
SHAPE = (20, 70, 5)


def same(run):
    for a, b in zip(*both_ways(run)):
        assert torch.equal(bits(a), bits(b))


@pytest.mark.parametrize("storage", ["f64", "f32", "f32dev", "f16dev", "bf16dev", "i16dev"])
@pytest.mark.parametrize("pattern", ["AA", "AB"])
@pytest.mark.parametrize("box", ["duct", "periodic"])
def test_step(storage, pattern, box):
    def run():
        g = lattice(*SHAPE, storage, pattern, duct(*SHAPE) if box == "duct" else None, True)
        assert box == "periodic" or 0 < 8 * g.d.row_count[0] <= SHAPE[0] * SHAPE[2]
        g.set_inflow(0.03, 0.0, 0.0)
        g.set_equilibrium_field(*fields(*SHAPE, 3))
        for t in range(4):
            g.step(output_macro=t == 3)
        torch.cuda.synchronize()
        return [d.clone() for d in g.df] + [g.macro.clone()]

    same(run)


@pytest.mark.parametrize("storage", ["f64", "f16dev"])
@pytest.mark.parametrize("pattern", ["AA", "AB"])
def test_coupled_step(storage, pattern):
    X, Y, Z = SHAPE
    ageo = np.full(SHAPE, ADE_GEO.FLUID, dtype=np.int16)
    ageo[:, :, 0] = ageo[:, :, -1] = ADE_GEO.WALL
    ageo[0] = ADE_GEO.INFLOW

    def run():
        g = lattice(X, Y, Z, storage, pattern, duct(X, Y, Z), True)
        a = D3Q7Lattice(g, collision="CLBM", diffusivity=0.0125, geo=ageo, phi_ref=0.0, store_scale=1000.0)
        assert 0 < 8 * a.d.row_count[0] <= X * Z
        g.set_inflow(0.03, 0.0, 0.0)
        g.set_equilibrium_field(*fields(X, Y, Z, 4))
        a.set_equilibrium(torch.tensor(np.random.default_rng(5).random((X, Y, Z)) * 1e-3))
        for t in range(4):
            g.step_coupled(a, output_macro=t == 3)
        torch.cuda.synchronize()
        return [d.clone() for d in g.df] + [d.clone() for d in a.df] + [g.macro.clone()]

    same(run)


@pytest.mark.parametrize("storage,tape", [("f64", None), ("f64", torch.float64), ("f64", torch.float32), ("f32", None),
                                          ("f32", torch.float32)])
def test_adjoint_step(storage, tape):
    """A periodic box: every slot is written by plain stores."""
    X, Y, Z = 6, 70, 5

    def run():
        g = D3Q27Lattice(X, Y, Z, storage=storage, pattern="AB", nu=0.02)
        g.set_equilibrium_field(*fields(X, Y, Z, 8))
        gen = torch.Generator(device="cuda").manual_seed(9)
        lam_next = torch.randn(g.df[0].numel(), generator=gen, device="cuda", dtype=g.df[0].dtype)
        lam = torch.zeros_like(lam_next)
        if tape is None:
            g.adjoint_step(lam_next, lam, None, which=0)
        else:
            rec = torch.zeros(tape_elements(g.d.XYZ), dtype=tape, device="cuda")
            f64 = int(tape == torch.float64)
            g._check(g.lib.tnl_lbm_d3q27_step_record(C.byref(g.cfg), C.byref(g.d), _ptr(rec), f64, _stream_ptr()))
            g._check(g.lib.tnl_lbm_d3q27_adjoint_step_recorded(C.byref(g.cfg), C.byref(g.d), _ptr(rec), f64,
                                                               _ptr(lam_next), _ptr(lam), None, _stream_ptr()))
        torch.cuda.synchronize()
        return [lam]

    same(run)
