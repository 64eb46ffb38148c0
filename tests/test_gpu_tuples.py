"""The sorted tuple list at the sizes where its two sorts meet: a star whose
centre has d leaves has d (d - 1) placements of a 3-vertex path through it,
plus none elsewhere; every list equals numpy's lexicographic order of the
same rows."""
import numpy as np
import pytest

from gpsm_amd import _lib
from gpsm_amd import graphs as G

pytestmark = pytest.mark.gpu


def star(leaves, n):
    """A star inside n vertices, its centre and leaves at scattered ids."""
    ids = np.random.default_rng(leaves).permutation(n)[:leaves + 1]
    return G.from_edges(n, np.full(leaves, ids[0]), ids[1:], np.ones(n)), ids


@pytest.mark.parametrize("leaves", [1, 2, 8, 64, 90, 91, 92, 300])  # 91 * 90 = 8190 rows, 92 * 91 = 8372
@pytest.mark.parametrize("n", [400, 70_000])
def test_rows_sorted(ctx, leaves, n):
    g, ids = star(leaves, n)
    r = ctx.upload(g).match(G.path_query(3), want_tuples=True, tuple_cap=1 << 17)
    a, b = np.meshgrid(ids[1:], ids[1:], indexing="ij")
    rows = np.stack([a.ravel(), np.full(a.size, ids[0]), b.ravel()], axis=1)[a.ravel() != b.ravel()]
    want = rows[np.lexsort(rows.T[::-1])].astype(np.uint32)
    assert r.count == len(want) == leaves * (leaves - 1)
    assert np.array_equal(r.tuples, want)


@pytest.mark.parametrize("cap", [1, 719, 720, 721])
def test_cap(ctx, cap):
    """720 placements of a 6-clique: a cap below them is an overflow."""
    rg = ctx.upload(G.complete(6))
    if cap < 720:
        with pytest.raises(_lib.GpsmError) as e:
            rg.match(G.clique_query(6), want_tuples=True, tuple_cap=cap)
        assert e.value.code == -5
    else:
        t = rg.match(G.clique_query(6), want_tuples=True, tuple_cap=cap).tuples
        assert t.shape == (720, 6) and np.array_equal(t, t[np.lexsort(t.T[::-1])])


def test_wide_rows(ctx):
    """Rows of 64 columns, whose packed number spans several 64-bit parts."""
    rg = ctx.upload(G.cycle(64))
    t = rg.match(G.path_query(64), want_tuples=True, tuple_cap=1000).tuples
    assert t.shape == (128, 64) and np.array_equal(t, t[np.lexsort(t.T[::-1])])
    rows = {tuple(x) for x in t.tolist()}
    assert len(rows) == 128 and tuple(range(64)) in rows


def test_list_outlives_the_result(ctx):
    rg = ctx.upload(G.complete(6))
    lists = [rg.match(G.clique_query(4), want_tuples=True, tuple_cap=1000).tuples for _ in range(50)]
    for t in lists[1:]:
        assert np.array_equal(t, lists[0])
    tail = lists[0][-1:]
    del lists
    assert tail.tolist() == [[5, 4, 3, 2]]
