"""Counting the last one or two join levels from per-candidate records
against enumerating them: a query matched for its count, the same query with
its tuples wanted (every embedding enumerated) and the oracle give the same
count, hash, rows and work per level, for every shape the last two positions
can take, on graphs whose few labels make the injectivity checks bite."""
import itertools

import numpy as np
import pytest

import pyoracle as O
from gpsm_amd import _lib
from gpsm_amd import graphs as G

pytestmark = pytest.mark.gpu

# edges of the query shapes; "y" and "w" are the last two vertices bound
SHAPES = {
    "edge": (2, [(0, 1)]),
    "path3": (3, [(0, 1), (1, 2)]),
    "path4": (4, [(0, 1), (1, 2), (2, 3)]),
    "star4": (4, [(0, 1), (0, 2), (0, 3)]),
    "path5": (5, [(0, 1), (1, 2), (2, 3), (3, 4)]),
    "fork5": (5, [(0, 1), (1, 2), (1, 3), (3, 4)]),
    "star6": (6, [(0, 1), (0, 2), (0, 3), (0, 4), (0, 5)]),
    "path6": (6, [(0, 1), (1, 2), (2, 3), (3, 4), (4, 5)]),
    "triangle": (3, [(0, 1), (1, 2), (0, 2)]),
    "tail4": (4, [(0, 1), (1, 2), (0, 2), (2, 3)]),
    "tails5": (5, [(0, 1), (1, 2), (0, 2), (2, 3), (2, 4)]),
    "chain5": (5, [(0, 1), (1, 2), (0, 2), (2, 3), (3, 4)]),
}


def orders(n, edges, rng, most=6):
    adj = [set() for _ in range(n)]
    for a, b in edges:
        adj[a].add(b)
        adj[b].add(a)
    out = [p for p in itertools.permutations(range(n))
           if all(adj[p[i]] & set(p[:i]) for i in range(1, n))]
    return [out[i] for i in rng.permutation(len(out))[:most]]


@pytest.mark.parametrize("labels", [1, 2, 3])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_counted_equals_enumerated_and_oracle(ctx, shape, labels):
    n, edges = SHAPES[shape]
    rng = np.random.default_rng(1000 * labels + len(shape))
    size = 700 if n <= 4 else 150
    g = G.small_graph(50 + labels, n=size, m=5 * size if n <= 4 else 3 * size, labels=labels, kind="cl")
    src, dst = (np.array(x, dtype=np.uint32) for x in zip(*edges))
    q = G.Query(rng.integers(1, labels + 1, size=n).astype(np.uint32), src, dst)
    try:
        ctx.set_hub_policy(6, 1 << 30)  # most edge tests through hub bitmaps, some by search
        rh = ctx.upload(g)
        ctx.set_hub_policy(512, 0)  # every edge test by search
        rn = ctx.upload(g)
    finally:
        ctx.set_hub_policy()
    for od in orders(n, edges, rng):
        ref = O.o2_match(g, q, mode=0, order=list(od))
        if ref["count"] > 3_000_000:
            continue
        full = rh.match(q, order_mode=_lib.ORDER_EXPLICIT, explicit_order=od, want_tuples=True, tuple_cap=4_000_000)
        assert len(full.tuples) == full.count == ref["count"]
        want = (full.count, full.hash, full.level_rows, full.level_work, full.join_work)
        for rg in (rh, rn):
            r = rg.match(q, order_mode=_lib.ORDER_EXPLICIT, explicit_order=od)
            assert (r.count, r.hash, r.level_rows, r.level_work, r.join_work) == want, (od, rg is rh)
        if ref["count"]:
            assert full.level_rows[1:] == ref["level_rows"][1:n] and full.hash == ref["hash"]


def test_counted_levels_keep_the_budget_exact(ctx):
    """The work of levels counted from records counts towards the budget as
    if they were enumerated."""
    g = G.small_graph(61, n=2000, m=16000, labels=2, kind="cl")
    rg = ctx.upload(g)
    for q in (G.path_query(4), G.star_query(3)):
        r = rg.match(q)
        assert r.join_work > r.level_work[1]
        assert rg.match(q, work_budget=r.join_work).count == r.count
        with pytest.raises(_lib.GpsmError) as e:
            rg.match(q, work_budget=r.join_work - 1)
        assert e.value.code == _lib.EBUDGET


def test_hub_rows_of_thousands_of_candidates(ctx):
    """Lists longer than one wave step and tables of more than one chunk of 64
    candidates, all vertices of one label: closed forms on a star of stars."""
    hubs, leaves = 5, 3000
    src = np.concatenate([np.zeros(hubs, dtype=np.uint32), np.repeat(np.arange(1, hubs + 1), leaves)])
    dst = np.concatenate([np.arange(1, hubs + 1), hubs + 1 + np.arange(hubs * leaves)])
    g = G.from_edges(1 + hubs + hubs * leaves, src, dst, np.ones(1 + hubs + hubs * leaves))
    rg = ctx.upload(g)
    deg = g.degree()
    paths = 0  # 4-vertex paths: ordered edge in the middle, one more neighbour at each end (no triangles here)
    for v in range(g.n):
        for w in g.col[g.row_offset[v]:g.row_offset[v + 1]]:
            paths += int(deg[v] - 1) * int(deg[w] - 1)
    assert rg.match(G.path_query(4)).count == paths
    assert rg.match(G.star_query(3)).count == int((deg * (deg - 1) * (deg - 2)).sum())
    assert rg.match(G.path_query(3)).count == int((deg * (deg - 1)).sum())
