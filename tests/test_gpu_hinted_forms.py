"""The kernels with cache hints and whole-line row shapes, which a step takes on large
arrays only, against the ones that small arrays take: a lattice that repeats a small one
along x steps as the small one does, tile by tile.  The sizes are checked against the
rule's constants in the source, so that a moved line does not leave them unreached.
Tolerance as for the row lists: 16 epsilons of an array's scale, one for stored 2-byte
values.  Also the paired even step of a map in rows (overlaps in y)."""
import ctypes as C
import re
from pathlib import Path

import numpy as np
import pytest
import torch

from pytnl_lbm import ADE_GEO, D3Q7Lattice
from pytnl_lbm._abi import GEO
from pytnl_lbm.adjoint import tape_elements
from pytnl_lbm.lattice import _ptr, _stream_ptr
from test_gpu_lean import geometry
from test_gpu_row_lists import fields, lattice, units, within

pytestmark = pytest.mark.gpu

SOURCE = (Path(__file__).resolve().parent.parent / "tnl-lbm_amd" / "csrc" / "lbm_step.hpp").read_text()
LLC = int(re.search(r"LLC_BYTES = (\d+)ull << 20", SOURCE).group(1)) << 20
TIMES = int(re.search(r"return bytes <= (\d+) \* LLC_BYTES;", SOURCE).group(1))
MEET = [int(m) << 20 for m in re.findall(r"A\.plane_bytes == (\d+)ull << 20", SOURCE)]

TILE = 8  # x planes of the small lattice
BYTES = {"f64": 8, "f32": 4, "f32dev": 4, "f16dev": 2, "bf16dev": 2, "i16dev": 2}
# x planes of the large one: A-A beyond the rule's size (256 x 256 planes; 27 or, with the scalar, 34 population
# planes), A-B on planes of 8 MiB (128 x 128 and 256 x 256)
AA = {8: 104, 4: 200, 2: 400}
AA_COUPLED = {8: 80, 4: 160, 2: 320}
AB = {8: (64, 128), 4: (128, 128), 2: (64, 256)}


def sizes(storage, pattern, planes):
    """(X, Y = Z) of the large lattice, one that takes hints where the small one does not."""
    e = BYTES[storage]
    X, Y = ((AA if planes == 27 else AA_COUPLED)[e], 256) if pattern == "AA" else AB[e]
    plane = X * Y * Y * e
    assert planes * plane > TIMES * LLC if pattern == "AA" else plane in MEET
    assert planes * (plane // X * TILE) <= TIMES * LLC and plane // X * TILE not in MEET and X % TILE == 0
    return X, Y


def tile(kind, Y, wall, inflow, periodic, sym=None):
    """Codes of the small lattice.  Only PERIODIC sites on its x faces: others pull from a
    clamped column there, which is not a face of the large lattice."""
    geo = np.full((TILE, Y, Y), periodic, dtype=np.int16)
    geo[1:-1, :, 0] = geo[1:-1, :, -1] = wall
    if kind == "few":
        geo[2, 1:-1, 2] = inflow
        geo[4, Y // 2, 3] = sym
    return geo


def repeat(big, small):
    """Each population plane of `big` (n planes of flat sites) as copies of `small`'s."""
    n = 27 if small.numel() % 27 == 0 else 7
    big.view(n, -1, small.numel() // n).copy_(small.view(n, 1, -1))


def same_tiles(tag, big, small, n):
    """Plane by plane, every tile of `big` within the tolerance of `small`."""
    tiles = big.view(n, -1, small.numel() // n)
    for k in range(n):
        s = small.view(n, 1, -1)[k]
        scale = small if small.dtype.is_floating_point else s
        full = s.expand_as(tiles[k])
        if small.dtype.is_floating_point:
            limit = (1.0 if small.element_size() == 2 else 16.0) * torch.finfo(small.dtype).eps * float(scale.double().abs().max())
            worst = float((tiles[k].double() - full.double()).abs().max())
        else:
            limit, worst = 1, int((tiles[k].int() - full.int()).abs().max())
        assert worst <= limit, (tag, k, worst, limit)


def pair(storage, pattern, kind, planes, lists=True):
    X, Y = sizes(storage, pattern, planes)
    geo = None if kind == "periodic" else tile(kind, Y, GEO.WALL, GEO.INFLOW, GEO.PERIODIC, GEO.SYM_TOP)
    small = lattice(TILE, Y, Y, storage, pattern, geo, lists)
    big = lattice(X, Y, Y, storage, pattern, None if geo is None else np.tile(geo, (X // TILE, 1, 1)), lists,
                  placement="first")
    small.set_equilibrium_field(*fields(TILE, Y, Y, 3))
    for lat in (small, big):
        lat.set_inflow(0.02, 0.0, 0.01)
    return small, big


@pytest.mark.parametrize("storage", list(BYTES))
@pytest.mark.parametrize("pattern,kind,lists", [("AA", "periodic", True), ("AA", "walls", True), ("AA", "few", True),
                                                ("AB", "walls", True), ("AB", "few", True), ("AB", "walls", False)])
def test_step(storage, pattern, kind, lists):
    small, big = pair(storage, pattern, kind, 27, lists)
    for t in range(2):
        for b, s in zip(big.df, small.df):
            repeat(b, s)
        for lat in (small, big):
            lat.step(output_macro=t == 1)
        torch.cuda.synchronize()
        for b, s in zip(big.df, small.df):
            same_tiles((storage, pattern, kind, t), b, s, 27)
    same_tiles((storage, pattern, kind, "macro"), big.macro, small.macro, 4)


@pytest.mark.parametrize("lists", [True, False])
@pytest.mark.parametrize("pattern", ["AA", "AB"])
@pytest.mark.parametrize("storage", ["f64", "f16dev"])
def test_coupled_step(storage, pattern, lists):
    small, big = pair(storage, pattern, "walls", 34, lists)
    scalars = []
    for lat in (small, big):
        ageo = np.tile(tile("walls", lat.Y, ADE_GEO.WALL, 0, ADE_GEO.PERIODIC), (lat.X // TILE, 1, 1))
        scalars.append(D3Q7Lattice(lat, collision="CLBM", diffusivity=0.02, geo=ageo, phi_ref=0.1, store_scale=50.0))
    a, b = scalars
    a.set_equilibrium(torch.as_tensor(0.1 + 0.01 * np.random.default_rng(6).random((small.X, small.Y, small.Z))))
    for t in range(2):
        for x, y in zip(big.df + b.df, small.df + a.df):
            repeat(x, y)
        small.step_coupled(a, output_macro=t == 1)
        big.step_coupled(b, output_macro=t == 1)
        torch.cuda.synchronize()
        for x, y in zip(big.df + b.df, small.df + a.df):
            same_tiles((storage, pattern, t), x, y, 27 if y.numel() % 27 == 0 else 7)
    same_tiles((storage, pattern, "phi"), b.phi, a.phi, 1)


@pytest.mark.parametrize("storage,tape", [("f64", torch.float64), ("f64", torch.float32), ("f32", torch.float32),
                                          ("from f64", torch.float32)])
def test_recording_step(storage, tape):
    small, big = pair("f32" if storage == "from f64" else storage, "AB", "few", 27)
    tapes = []
    for lat in (small, big):
        if lat is big:
            repeat(big.df[0], small.df[0])
        rec = torch.zeros(tape_elements(lat.d.XYZ), dtype=tape, device="cuda")
        if storage == "from f64":
            state = lat.df[0].double()
            lat._check(lat.lib.tnl_lbm_d3q27_step_record_from_f64(C.byref(lat.cfg), C.byref(lat.d), _ptr(state), _ptr(rec),
                                                                  _stream_ptr()))
        else:
            lat._check(lat.lib.tnl_lbm_d3q27_step_record(C.byref(lat.cfg), C.byref(lat.d), _ptr(rec),
                                                         int(tape == torch.float64), _stream_ptr()))
        tapes.append(rec)
    torch.cuda.synchronize()
    same_tiles((storage, tape), big.df[1], small.df[1], 27)
    # blocks of 64 sites, so tiles of whole blocks
    same_tiles((storage, tape, "recording"), tapes[1], tapes[0], 1)


@pytest.mark.parametrize("storage", ["f16dev", "bf16dev", "i16dev"])
def test_pairs_of_a_map_in_rows(storage):
    """Few rows with walls, overlaps in y: the even step takes pairs of sites row by row."""
    X, Y, Z, o = 4, 70, 20, (1, 2, 1)
    geo = geometry("walls", X, Y, Z)
    geo[1, 7, 5] = geo[2, 12, 9] = GEO.WALL  # one site of a pair
    geo[3, 9, 11] = GEO.INFLOW
    a, b = (lattice(X, Y, Z, storage, "AA", geo, rl, overlap=o) for rl in (True, False))
    assert a.d.row_count[2] * 8 <= X * Z and 0 < a.d.row_count[0] * 8 <= X * Z
    stored = tuple(n + 2 * k for n, k in zip((X, Y, Z), o))
    c = lattice(*stored, storage, "AA", None, False)
    c.set_equilibrium_field(*fields(*stored, 5))
    force = [1e-5 * np.random.default_rng(2).standard_normal(stored) for _ in range(3)]
    for lat in (a, b):
        lat.set_force_field(*force)
        lat.set_inflow(0.02, 0.0, 0.01)
    for t in range(4):
        for lat in (a, b):
            lat.df[0].copy_(c.df[0])
            lat.step(output_macro=t > 1)
        torch.cuda.synchronize()
        for x, y in ((a.df[0], b.df[0]), (a.macro, b.macro)):
            assert within(x, y), (storage, t, units(x, y))
