"""The x-slab halo exchange moves exactly its planes: every slot of the stored
lattices against slices of the arrays before it, over plane sizes and bases of
every alignment (16, 8, 4 and 2 bytes), ends of the copy's 8 KB pieces, one
slab that is its own neighbour, two slabs, and an exchange inside a captured
graph."""
import pytest
import torch

from lbm_common import CX
from pytnl_lbm import D3Q27Lattice, _abi

pytestmark = pytest.mark.gpu


def slab(X, Y, Z, storage, pattern, overlap, seed):
    lat = D3Q27Lattice(X, Y, Z, storage=storage, pattern=pattern, nu=0.01, overlap=overlap)
    g = torch.Generator().manual_seed(seed)
    raw = torch.randint(0, 255, (lat.df[0].numel() * lat.df[0].element_size(),), generator=g, dtype=torch.uint8)
    lat.df[0].copy_(raw.view(lat.df[0].dtype))
    return lat


def bits(lat):
    # bytes as a trailing axis: (q, x, z, y, byte)
    t = lat.stored(0).contiguous()
    return t.view(torch.uint8).view(*t.shape, t.element_size()).clone()


def expected(lo, up, phase, aa):
    before = {lo: bits(lo), up: bits(up)}
    after = {lat: b.clone() for lat, b in before.items()}
    for q in range(27):
        if CX[q] == 0:
            continue
        # (ghost plane, the boundary plane it mirrors)
        if (CX[q] > 0) == aa:
            ghost, edge = (lo, lo.ox + lo.X), (up, up.ox)
        else:
            ghost, edge = (up, up.ox - 1), (lo, lo.ox + lo.X - 1)
        dst, src = (ghost, edge) if phase == _abi.HALO_PULL else (edge, ghost)
        after[dst[0]][q, dst[1]] = before[src[0]][q, src[1]]
    return after[lo], after[up]


@pytest.mark.parametrize("storage", ["f64", "f32", "f16dev"])
@pytest.mark.parametrize("Y,Z,X", [(7, 3, 1), (64, 32, 2), (128, 8, 3), (129, 17, 2), (67, 61, 1), (512, 9, 2), (1, 1, 2)])
def test_exchange_moves_exactly_its_planes(Y, Z, X, storage):
    for pattern, phases in (("AA", (_abi.HALO_PULL, _abi.HALO_PUSH)), ("AB", (_abi.HALO_PULL,))):
        for phase in phases:
            for two in (False, True):
                lo = slab(X, Y, Z, storage, pattern, (1, 0, 0), 1)
                up = slab(X + 1, Y, Z, storage, pattern, (2, 0, 0), 2) if two else lo
                ref = expected(lo, up, phase, pattern == "AA")
                lo.halo_x(up, phase)
                torch.cuda.synchronize()
                for lat, r in zip((lo, up), ref):
                    assert torch.equal(bits(lat), r), (pattern, phase, two)


def test_exchange_in_a_captured_graph():
    """Recorded and replayed with eager work in between, as the eager exchange."""
    lo = slab(3, 96, 40, "f64", "AA", (1, 1, 1), 3)
    ref = expected(lo, lo, _abi.HALO_PULL, True)[0]
    start = lo.df[0].clone()
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        lo.halo_x(lo, _abi.HALO_PULL)
    for _ in range(3):
        lo.df[0].copy_(start)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(bits(lo), ref)
