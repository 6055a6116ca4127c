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


@pytest.mark.parametrize("name", ["rod", "ties", "pair_of_columns"])
def test_grid_order_of_long_columns_and_ties(name):
    # a column beyond the LDS sort, atoms at equal z (and at 0 and -0), and
    # odd column lengths: the order is (z, index), as the oracle's
    print(f"[grid] {name}", flush=True)
    rng = np.random.default_rng(7)
    if name == "rod":
        x = rng.uniform(0, 1, (3001, 3)) * [0.1, 0.1, 5.0]
    elif name == "ties":
        x = rng.integers(0, 24, (1500, 3)) * 0.2 + rng.uniform(0, 0.01, (1500, 3)) * [1, 1, 0]
        x[:3, 2] = 0.0
    else:
        x = rng.uniform(0, 1, (7, 3)) * 4.9
    n = len(x)
    s = S.System(name, np.full(3, 5.0), S._wrap(x, np.full(3, 5.0)), np.zeros(n, np.int32), np.zeros(n),
                 np.array([1e-3]), np.array([1e-6]), np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32),
                 0.3, 0.3)
    ctx = nbx.Context(rlist=s.rlist)
    ctx.set_nonbonded_parameters(*nbx.nblib_c6c12_matrices(s.c6, s.c12))
    ctx.set_topology(s.types, s.charges, s.excl_off, s.excl_idx)
    x32 = s.x.astype(np.float32)
    x32[1, 2] *= -1.0 if name == "ties" else 1.0  # -0
    ctx.put_on_grid(s.box, x32)
    g = oracle_for(s, "f32").grid()
    ai, cells = ctx.grid()
    np.testing.assert_array_equal(ai, g["atomIndices"])
    np.testing.assert_array_equal(cells, g["cells"])


def test_rebuilt_layout_equals_the_first(monkeypatch):
    # the first search counts before it writes; later ones leave the list in
    # regions that the group pass makes compact: the same layout either way,
    # and from the pruned list at the full radius
    s = S.water_box(1501, None, seed=12, rc=0.9, rlist=1.0)
    for sort in ("0", "1"):
        monkeypatch.setenv("NBX_UNION_SORT", sort)
        ctx = nbx.context_for(s)
        layouts = [ctx.work_groups()]
        ctx.put_on_grid(s.box, s.x)
        ctx.construct_pairlist()
        layouts.append(ctx.work_groups())
        f = ctx.compute(s.x)
        ctx.prune_pairlist(1.0)
        layouts.append(ctx.work_groups())
        for other in layouts[1:]:
            for key in ("groups", "chunks", "union", "work"):
                np.testing.assert_array_equal(layouts[0][key], other[key], err_msg=key)
        np.testing.assert_array_equal(f, ctx.compute(s.x))
