"""The periodic A-A steps over boxes whose rows do not fill blocks or lines: the
even step's flat range against its rows (a box split into sub-box launches
steps the same sites through the other mapping), the odd step's linear mapping
against whole rows, and a slab whose overlaps leave a flat range that does not
start at the array; F64 against the oracle."""
import numpy as np
import pytest
import torch

import oracle as O
from lbm_common import W, rel_max
from pytnl_lbm import D3Q27Lattice, _abi

pytestmark = pytest.mark.gpu

# rows below a wave, between waves and blocks, one over a block, whole blocks;
# even and odd site counts (pairs of 2-byte sites, plane alignment)
SHAPES = [(1, 1, 1), (3, 2, 5), (5, 30, 7), (3, 63, 5), (4, 65, 6), (7, 97, 3), (2, 127, 9), (3, 187, 4), (2, 257, 3),
          (2, 320, 2), (3, 513, 2), (2, 256, 4), (1, 512, 3)]
FORMS = ["f64", "f32", "f32dev", "f16dev", "bf16dev", "i16dev"]


def lattice(shape, storage, seed, **kw):
    lat = D3Q27Lattice(*shape, storage=storage, nu=0.01, store_range=0.5, **kw)
    rng = np.random.default_rng(seed)
    n = lat.nsites
    f = torch.as_tensor(0.02 * rng.standard_normal((27, n)))
    dev = f * torch.as_tensor(W)[:, None]
    dst = lat.df[0].view(27, lat.d.XYZ)[:, :n]
    if storage == "i16dev":
        dst.copy_((f / 0.5 * 32767).round().to(torch.int16))
    else:
        dst.copy_(dev if storage.endswith("dev") else dev + torch.as_tensor(W)[:, None])
    return lat


def step_in_pieces(lat):
    """One step as launches over sub-boxes split in every axis."""
    cuts = [sorted({0, n // 3, n}) for n in (lat.X, lat.Y, lat.Z)]
    t = lat.iterations
    for x in zip(cuts[0], cuts[0][1:]):
        for y in zip(cuts[1], cuts[1][1:]):
            for z in zip(cuts[2], cuts[2][1:]):
                lat.iterations = t
                lat.step(offset=(x[0], y[0], z[0]), end=(x[1], y[1], z[1]))


def close(a, b, storage):
    """The mappings run the same operations; fused multiplies and adds may
    differ between the kernels: 8 epsilons of the array's scale, one unit of a
    2-byte form's stored value (its rounding may flip)."""
    if a.dtype == torch.int16:
        return int((a.int() - b.int()).abs().max()) <= 1
    x, y = a.double(), b.double()
    if a.element_size() == 2:
        ulp = 2.0 ** (torch.floor(torch.log2(y.abs().clamp_min(1e-7))) - (10 if a.dtype == torch.float16 else 7))
        return bool(((x - y).abs() <= ulp + 1e-7).all())
    return float((x - y).abs().max()) <= 8 * torch.finfo(a.dtype).eps * float(y.abs().max())


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("storage", FORMS)
def test_whole_box_equals_its_sub_boxes(shape, storage):
    a, b = lattice(shape, storage, 3), lattice(shape, storage, 3)
    for _ in range(2):  # one even and one odd step, each from the same state
        a.step(output_macro=False)
        step_in_pieces(b)
        torch.cuda.synchronize()
        assert close(a.df[0], b.df[0], storage), (shape, storage, a.iterations)
        b.df[0].copy_(a.df[0])


@pytest.mark.parametrize("storage,shape", [("f64", (80, 256, 64)), ("f64", (60, 208, 110)), ("f16dev", (200, 256, 100)),
                                           ("f32", (100, 512, 50))])
def test_boxes_beyond_the_cache(storage, shape):
    """Populations above the last-level cache, planes on lines: the forms with hints."""
    test_whole_box_equals_its_sub_boxes(shape, storage)


@pytest.mark.parametrize("shape", [(3, 63, 5), (7, 97, 3), (2, 320, 2), (3, 513, 2)])
def test_f64_against_the_oracle(shape):
    a = lattice(shape, "f64", 5)
    h = O.HostLattice(*shape, pattern=_abi.PATTERN_AA, nu=0.01)
    h.import_f64(a.export_f64(0).cpu().numpy(), which=0)
    for _ in range(4):
        a.step(output_macro=True)
        h.step(output_macro=True)
    got, ref = a.export_f64(0).cpu().numpy(), h.export_f64(0)
    assert rel_max(got, ref) < 4e-13  # 1e-13 a step
    for x, y in zip(a.macros(), h.macros()):
        assert np.abs(x.cpu().numpy() - y).max() < 4e-13


@pytest.mark.parametrize("storage", ["f64", "f16dev"])
@pytest.mark.parametrize("overlap", [(1, 0, 0), (1, 1, 1)])
def test_slab_matches_the_periodic_box(storage, overlap):
    """A self-periodic slab's even step touches its own sites only: the sites of
    a lattice with overlaps step as those of the box, the ghosts keep theirs."""
    shape = (5, 46, 7)
    a, b = lattice(shape, storage, 9), lattice(shape, storage, 9, overlap=overlap, XYZ=(shape[0] + 2 * overlap[0])
                                               * (shape[1] + 2 * overlap[1]) * (shape[2] + 2 * overlap[2]))
    ox, oy, oz = overlap
    inner = b.stored()[:, ox:ox + shape[0], oz:oz + shape[2], oy:oy + shape[1]]
    b.df[0].fill_(0)
    inner.copy_(a.df[0].view(27, shape[0], shape[2], shape[1]))
    before = b.df[0].clone()
    a.step()
    b.step()
    torch.cuda.synchronize()
    got = inner.reshape(-1)
    assert close(got, a.df[0], storage)
    inner.copy_(before.view(b.stored().shape)[:, ox:ox + shape[0], oz:oz + shape[2], oy:oy + shape[1]])
    assert torch.equal(b.df[0], before)
