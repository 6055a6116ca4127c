"""The search where its candidate lists are long or uneven."""
import numpy as np
import pytest

from gmxapi_amd import nbx, systems as S
from oracle import oracle as O
from tests.helpers import oracle_for

pytestmark = pytest.mark.gpu


def _dense_corner(n, box, edge, rlist, seed):
    """n atoms in a cube of the given edge at the corner of a larger box: few
    grid columns, each with many clusters, and most columns empty."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    k = np.arange(n)
    x = (np.stack([k // (m * m), (k // m) % m, k % m], 1) + 0.5) * (edge / m) + rng.uniform(-0.02, 0.02, (n, 3))
    off = np.arange(n + 1, dtype=np.int32)
    x = S._wrap(x, np.full(3, box))
    return S.System("corner", np.full(3, box), x, np.zeros(n, np.int32), np.zeros(n), np.array([1e-3]),
                    np.array([1e-6]), off, off[:-1].copy(), rlist, rlist)


@pytest.mark.parametrize("n,box,edge,rlist", [
    (3000, 6.0, 1.9, 0.9),   # more than 512 candidates in a window of columns
    (257, 2.3, 2.29, 1.1),   # every cluster reaches through every face
    (5, 2.4, 0.6, 1.2),      # a partly filled cluster, one column
    (20000, 5.2, 5.19, 1.3), # more than 64 columns in range
])
def test_pair_set_of_uneven_systems(n, box, edge, rlist):
    print(f"[search] {n} atoms in {edge} of {box} nm, rlist {rlist}", flush=True)
    s = _dense_corner(n, box, edge, rlist, seed=n)
    ctx = nbx.context_for(s)
    want = O.brute_pairs(s.x, s.box, s.rlist, "f32") if n <= 3000 else oracle_for(s, "f32").list_pairs(s.rlist)
    first = ctx.pairlist()
    np.testing.assert_array_equal(ctx.list_pairs(s.rlist), want)
    # the second search writes without a count pass
    ctx.put_on_grid(s.box, s.x)
    ctx.construct_pairlist()
    for a, b in zip(first, ctx.pairlist()):
        np.testing.assert_array_equal(a, b)
