"""Sorted tuple lists whose rows' packed bits end just below and above one and
two 64-bit parts: paths of q vertices around a cycle with scattered ids."""
import numpy as np
import pytest

from gpsm_amd import graphs as G

pytestmark = pytest.mark.gpu


# 9 bits a vertex: 63, 72, 126 and 135 bits; 13 bits: 65, 117 and 130
@pytest.mark.parametrize("n,q", [(400, 7), (400, 8), (400, 14), (400, 15), (5000, 5), (5000, 9), (4200, 10)])
def test_path_rows_sorted(ctx, n, q):
    ids = np.random.default_rng(n + q).permutation(n).astype(np.uint32)
    g = G.from_edges(n, ids, np.roll(ids, 1), np.ones(n))
    t = ctx.upload(g).match(G.path_query(q), want_tuples=True, tuple_cap=1 << 14).tuples
    rows = np.stack([np.roll(ids, -j) for j in range(q)], axis=1)
    rows = np.concatenate([rows, rows[:, ::-1]])
    assert np.array_equal(t, rows[np.lexsort(rows.T[::-1])])


@pytest.mark.parametrize("q", [4, 5])
def test_rows_with_common_columns(ctx, q):
    """A vertex of 40 arms on 70,000 vertices (17 bits a column: 68 and 85
    bits): rows that agree in all but the last columns."""
    n, arms = 70_000, 40
    ids = np.random.default_rng(q).permutation(n).astype(np.uint32)
    a, b = ids[1:1 + arms], ids[1 + arms:1 + 2 * arms]
    g = G.from_edges(n, np.concatenate([np.full(arms, ids[0]), a]), np.concatenate([a, b]), np.ones(n))
    t = ctx.upload(g).match(G.path_query(q), want_tuples=True, tuple_cap=1 << 13).tuples
    assert len(t) == 2 * arms * (arms - 1) if q == 4 else len(t) == arms * (arms - 1)
    assert np.array_equal(t, t[np.lexsort(t.T[::-1])])
    assert len(np.unique(t, axis=0)) == len(t)
