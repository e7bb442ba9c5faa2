"""The recording step from an FP64 state against the conversion of the state to
F32 followed by the F32 recording step: the same populations and the same
recording, bit for bit, over row lengths around the waves and blocks, every
geometry code with an adjoint, both slot addressings and a hinted size."""
import ctypes as C

import pytest
import torch

from pytnl_lbm import GEO, D3Q27Lattice, _abi
from pytnl_lbm.adjoint import tape_elements
from pytnl_lbm.lattice import _ptr, _stream_ptr

pytestmark = pytest.mark.gpu


def geometry(kind, X, Y, Z):
    geo = torch.full((X, Y, Z), GEO.PERIODIC if kind == "periodic" else GEO.FLUID, dtype=torch.int16)
    if kind != "periodic":
        geo[:, 0] = geo[:, -1] = geo[:, :, 0] = geo[:, :, -1] = GEO.WALL
        geo[0] = GEO.INFLOW
        geo[-1] = GEO.OUTFLOW_RIGHT if kind == "right" else GEO.OUTFLOW_EQ
        geo[X // 2, Y // 2, Z // 2] = GEO.NOTHING
    return geo


@pytest.mark.parametrize("kind", ["periodic", "right", "eq"])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("shape", [(3, 5, 4), (4, 64, 3), (5, 65, 7), (3, 128, 5), (2, 257, 3), (160, 64, 128)])
def test_equals_conversion_and_step(shape, wide, kind):
    X, Y, Z = shape
    lat = D3Q27Lattice(X, Y, Z, storage="f32", pattern="AB", nu=0.01, geo=geometry(kind, X, Y, Z), force=(1e-5, 0, -2e-6))
    g = torch.Generator(device="cuda").manual_seed(X + Y)
    v = torch.rand(3, Z, Y, generator=g, device="cuda", dtype=torch.float64) * 0.05
    lat.set_inflow(profile=[v[0], v[1], v[2]])
    lat.set_equilibrium(1.0, 0.03, -0.02, 0.01)
    state = lat.df[0].double() * (1 + 0.01 * torch.rand(lat.df[0].shape, generator=g, device="cuda", dtype=torch.float64))
    n = tape_elements(lat.d.XYZ)
    out = []
    saved = lat.lib.tnl_lbm_set_wide_addressing(int(wide))
    try:
        for fused in (False, True):
            tape = torch.zeros(n, dtype=torch.float32, device="cuda")
            lat.df[1].zero_()
            lat._bind()
            if fused:
                lat._check(lat.lib.tnl_lbm_d3q27_step_record_from_f64(C.byref(lat.cfg), C.byref(lat.d), _ptr(state),
                                                                      _ptr(tape), _stream_ptr()))
            else:
                lat.df[0].copy_(state)
                lat._check(lat.lib.tnl_lbm_d3q27_step_record(C.byref(lat.cfg), C.byref(lat.d), _ptr(tape), 0, _stream_ptr()))
            torch.cuda.synchronize()
            out.append((lat.df[1].clone(), tape))
    finally:
        lat.lib.tnl_lbm_set_wide_addressing(saved)
    assert torch.equal(out[0][0].view(torch.int32), out[1][0].view(torch.int32))
    assert torch.equal(out[0][1].view(torch.int32), out[1][1].view(torch.int32))


def test_refuses_what_it_is_not_built_for():
    lat = D3Q27Lattice(4, 5, 3, storage="f64", pattern="AB", nu=0.01)
    t = torch.zeros(tape_elements(lat.d.XYZ), dtype=torch.float32, device="cuda")
    call = lat.lib.tnl_lbm_d3q27_step_record_from_f64
    assert call(C.byref(lat.cfg), C.byref(lat.d), _ptr(lat.df[0]), _ptr(t), _stream_ptr()) == _abi.ERR_UNSUPPORTED
    f32 = D3Q27Lattice(4, 5, 3, storage="f32", pattern="AB", nu=0.01)
    assert call(C.byref(f32.cfg), C.byref(f32.d), None, _ptr(t), _stream_ptr()) == _abi.ERR_NULL
    assert call(C.byref(f32.cfg), C.byref(f32.d), _ptr(lat.df[0]), _ptr(lat.df[0]), _stream_ptr()) == _abi.ERR_ARG
