"""A box without a geometry map and with a force field is stepped by the map kernels
as all PERIODIC, also with the row lists that tnl_lbm_classify_rows gives for it
(no map counts as all PERIODIC): every form and both parities, through the C entry
points, against the general kernel over a map of PERIODIC codes.  Tolerance as for
the row lists: 16 epsilons of an array's scale, one for stored 2-byte values."""
import numpy as np
import pytest
import torch

from pytnl_lbm._abi import GEO
from pytnl_lbm.lattice import classify_rows
from test_gpu_row_lists import fields, lattice, units, within

pytestmark = pytest.mark.gpu


# pairs of 2-byte sites over a flat range, odd rows (one site per lane), rows with overlaps
@pytest.mark.parametrize("shape,overlap", [((4, 70, 6), (0, 0, 0)), ((3, 33, 5), (0, 0, 0)), ((3, 70, 5), (1, 2, 1))])
@pytest.mark.parametrize("pattern", ["AA", "AB"])
@pytest.mark.parametrize("storage", ["f64", "f32", "f32dev", "f16dev", "bf16dev", "i16dev"])
def test_force_field_and_lists_without_a_map(storage, pattern, shape, overlap):
    X, Y, Z = shape
    a = lattice(X, Y, Z, storage, pattern, None, True, overlap=overlap)
    b = lattice(X, Y, Z, storage, pattern, np.full(shape, GEO.PERIODIC, dtype=np.int16), False, overlap=overlap)
    stored = tuple(n + 2 * o for n, o in zip(shape, overlap))
    force = [1e-5 * np.random.default_rng(2).standard_normal(stored) for _ in range(3)]
    for lat in (a, b):
        lat.set_force_field(*force)
    # some state, the same in both: equilibria of a field over the stored sites
    c = lattice(*stored, storage, pattern, None, False)
    c.set_equilibrium_field(*fields(*stored, 4))
    rows, counts = classify_rows(a, None)
    assert counts == (0, X * Z, 0) and a.d.map is None
    for t in range(4):
        for x, y, z in zip(a.df, b.df, c.df):
            x.copy_(z)
            y.copy_(z)
        a.d.rows = rows.data_ptr()
        for k in range(3):
            a.d.row_count[k] = counts[k]
        a.step(output_macro=t > 1)
        b.step(output_macro=t > 1)
        torch.cuda.synchronize()
        for x, y in zip(a.df + [a.macro], b.df + [b.macro]):
            assert within(x, y), (storage, pattern, shape, t, units(x, y))
