"""Every site is stepped once whatever the number of blocks: free streaming
through the periodic step kernels (bit for bit) on boxes whose block counts lie
around a power of two times the XCDs, where the size of the groups of blocks
changes, and at their remainders; an A-B step over the box against the same step
in parts, whose launches have other block counts."""
import pytest
import torch

from lbm_common import CX, CY, CZ, OPP
from pytnl_lbm import D3Q27Lattice

pytestmark = pytest.mark.gpu


# X Z rows of one 64-site block each: 1 to 257 blocks of arrays that the L2 caches
# hold, 4095 to 4097, 16 * 8 * 33 and 20000 of larger ones; then 32768 and 32769
# blocks of 512 two-byte sites, and more bytes than alternating order is taken for
@pytest.mark.parametrize("storage,shape", [("f32", (1, 64, n)) for n in (1, 7, 8, 9, 127, 128, 129, 255, 256, 257)]
                         + [("f32", (63, 64, 65)), ("f64", (63, 64, 65)), ("f64", (64, 64, 64)), ("f64", (17, 64, 241)),
                            ("f64", (66, 64, 64)), ("f32", (100, 64, 200)), ("f64", (61, 67, 71)), ("f16dev", (128, 512, 256)),
                            ("f16dev", (99, 512, 331)), ("f16dev", (203, 512, 256))])
def test_streaming_covers_the_box_once(storage, shape):
    X, Y, Z = shape
    g = D3Q27Lattice(X, Y, Z, storage=storage, nu=0.01)
    g.df[0].copy_(torch.arange(g.df[0].numel(), device="cuda") % 1013)  # exact in every form
    s0 = g.stored().clone()
    g.stream_only()
    torch.cuda.synchronize()
    for q in range(27):
        assert torch.equal(g.stored()[int(OPP[q])], s0[q]), ("even", q)
    g.stream_only()
    torch.cuda.synchronize()
    for q in range(27):
        want = torch.roll(s0[q], shifts=(2 * int(CX[q]), 2 * int(CZ[q]), 2 * int(CY[q])), dims=(0, 1, 2))
        assert torch.equal(g.stored()[q], want), ("odd", q)


@pytest.mark.parametrize("shape", [(5, 96, 40), (33, 64, 62), (64, 70, 33)])
def test_whole_step_equals_its_parts(shape):
    X, Y, Z = shape
    lats = [D3Q27Lattice(X, Y, Z, storage="f64", pattern="AB", nu=0.01) for _ in range(2)]
    gen = torch.Generator(device="cuda").manual_seed(3)
    f = None
    for lat in lats:
        lat.set_equilibrium(1.0, 0.02, -0.01, 0.03)
        if f is None:
            f = lat.df[0] * (1 + 0.01 * torch.rand(lat.df[0].shape, generator=gen, device="cuda", dtype=torch.float64))
        lat.df[0].copy_(f)
        lat.df[1].zero_()
    for lat in lats:
        lat.iterations = 1  # an odd step, from df[1]
        lat.df[1].copy_(f)
        lat.df[0].zero_()
    lats[0].step()
    cut = X // 3
    for k, (lo, hi) in enumerate(((0, cut), (cut, X))):
        lats[1].step(offset=(lo, 0, 0), end=(hi, Y, Z))
        lats[1].iterations -= 1 if k == 0 else 0
    torch.cuda.synchronize()
    assert torch.equal(lats[0].df[0], lats[1].df[0])
