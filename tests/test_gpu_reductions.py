"""The FP64 reductions over the macro field against numpy, at the edges of their
work splits: one site, rows and planes below and above a block, a plane of more
columns than blocks hold, ragged sizes, overlaps on each axis, distributed
axes, both element types, and NaN counts; several host threads at once.

The bound: n-term FP64 sums of the same terms in another order differ by at
most n eps times the sum of absolute values; the gradient terms are formed the
same way on both sides up to a few roundings (8 eps each)."""
import threading

import numpy as np
import pytest
import torch

from pytnl_lbm import D3Q27Lattice, _abi

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps
SHAPES = [(1, 1, 1), (5, 3, 4), (2, 64, 4), (9, 65, 63), (70, 16, 16), (3, 520, 513), (33, 47, 29), (1, 129, 2), (40, 5, 7)]


def lattice(shape, storage, overlap, seed):
    lat = D3Q27Lattice(*shape, storage=storage, nu=0.01, overlap=overlap)
    g = torch.Generator(device="cuda").manual_seed(seed)
    lat.macro.normal_(generator=g).mul_(0.05)
    lat.macro[:lat.d.XYZ] += 1
    X, Y, Z = (n + 2 * o for n, o in zip(shape, overlap))
    m = lat.macro.view(4, lat.d.XYZ)[:, :X * Y * Z].view(4, X, Z, Y).permute(0, 1, 3, 2)
    return lat, m.double().cpu().numpy()


def neighbours(a, axis, n, o, dist):
    """a at +1 and -1 along an axis, over the local sites."""
    i = np.arange(n)
    up, dn = i + 1, i - 1
    if not dist:
        up, dn = up % n, dn % n
    return a.take(up + o, axis), a.take(dn + o, axis)


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("overlap", [(0, 0, 0), (1, 0, 0), (1, 2, 1)])
@pytest.mark.parametrize("shape", SHAPES)
def test_sums_match_numpy(shape, overlap, storage):
    lat, m = lattice(shape, storage, overlap, 7)
    inner = tuple(slice(o, o + n) for n, o in zip(shape, overlap))
    rho, u = m[0][inner], m[1:][(slice(None),) + inner]
    n = rho.size
    u2 = (u ** 2).sum(0)
    got = lat.reduce_macro()
    for k, term in ((0, rho), (1, rho * u2), (3, (rho - 1) ** 2), (4, u2)):
        assert abs(got[k] - term.sum()) <= (n + 8) * EPS * np.abs(term).sum(), k
    assert got[2] == 0 and got[5] == n
    flags = (0,) if overlap == (0, 0, 0) else (0, _abi.FLAG_DISTRIBUTED_X)
    if overlap[1]:
        flags += (_abi.FLAG_DISTRIBUTED_X | _abi.FLAG_DISTRIBUTED_Y | _abi.FLAG_DISTRIBUTED_Z,)
    for fl in flags:
        dist = (fl & _abi.FLAG_DISTRIBUTED_X, fl & _abi.FLAG_DISTRIBUTED_Y, fl & _abi.FLAG_DISTRIBUTED_Z)
        G = np.empty((3, 3) + tuple(shape))
        for b in range(3):
            rest = (slice(None),) + tuple(slice(None) if a == b else inner[a] for a in range(3))
            up, dn = neighbours(m[1:][rest], b + 1, shape[b], overlap[b], dist[b])
            G[:, b] = 0.5 * (up - dn)
        w = np.stack([G[2, 1] - G[1, 2], G[0, 2] - G[2, 0], G[1, 0] - G[0, 1]])
        for g, term in zip(lat.reduce_gradients(flags=fl), (rho * (G ** 2).sum((0, 1)), rho * (w ** 2).sum(0))):
            # (the curl's differences cancel: its terms are bounded by 2 rho |G|^2)
            scale = 2 * np.abs(rho * (G ** 2).sum((0, 1))).sum()
            assert abs(g - term.sum()) <= (n + 16) * EPS * scale, fl
    # NaN densities are counted
    lat.macro[:lat.d.XYZ].view(-1)[((overlap[0]) * (shape[2] + 2 * overlap[2]) + overlap[2]) * (shape[1] + 2 * overlap[1])
                                   + overlap[1]] = float("nan")
    assert lat.reduce_macro()[2] == 1


def test_threads_reduce_at_once():
    """Each host thread gets its own lattice's sums."""
    lats = [lattice((24 + 3 * k, 33, 17), "f64", (0, 0, 0), k)[0] for k in range(6)]
    torch.cuda.synchronize()
    ref = [(lat.reduce_macro(), lat.reduce_gradients()) for lat in lats]
    bad = []

    def work(k):
        for _ in range(30):
            if (lats[k].reduce_macro(), lats[k].reduce_gradients()) != ref[k]:
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
