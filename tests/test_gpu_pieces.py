"""The device's numbering of the vertices by label and the adjacency's pieces
by the neighbours' label: numbers of labels around the groups a table of
pieces holds and the digits the entries are sorted by, empty labels' ranges at
vertex-range edges, graphs without edges, with and without hubs."""
import numpy as np
import pytest

import pyoracle as O
from gpsm_amd import _lib
from gpsm_amd import graphs as G

pytestmark = pytest.mark.gpu


def labelled(n, m, nl, seed):
    """Label values 3, 6, ... on a random graph, the first ones on half of it."""
    g = G.chung_lu(n, m, 2.1, seed)
    r = np.random.default_rng(seed)
    lab = r.permutation(np.concatenate([np.arange(nl), r.integers(0, nl, (n - nl) // 2),
                                        r.integers(0, min(nl, 3), n - nl - (n - nl) // 2)]))
    g.labels = (3 * (lab + 1)).astype(np.uint32)
    return g


def check(rg, g, q, tag):
    st, _, ref, _ = O.o2_filter(g, q)
    bm, cnt = rg.filter(q)
    if st == O.OK:
        for u in range(q.n):
            bits = np.unpackbits(bm[u].view(np.uint8), bitorder="little")[:g.n]
            assert np.array_equal(bits != 0, ref[u] != 0), (tag, u)
    r = O.o1_enumerate(g, q, tuple_cap=1 << 20)
    m = rg.match(q, want_tuples=True, tuple_cap=1 << 20)
    assert (m.count, m.hash) == (r["count"], r["hash"]), tag
    assert m.tuples.tobytes() == r["tuples"].tobytes(), tag
    b = rg.match_batch([q, q])
    assert [(x.count, x.hash) for x in b] == [(r["count"], r["hash"])] * 2, tag
    if st == O.OK and (cnt != 0).all():
        edges, tables = rg.candidate_edges(q)
        for (x, w), (ids, off, lst) in zip(edges, tables):
            assert np.array_equal(ids, np.flatnonzero(ref[x]))
            for i, v in enumerate(ids):
                nb = g.col[g.row_offset[v]:g.row_offset[v + 1]]
                assert np.array_equal(lst[off[i]:off[i + 1]], nb[ref[w][nb] != 0]), (tag, x, w, v)


# 64: the most groups; 65, 255 .. 257: labels share groups, one and two sorted
# digits; 4095: the most labels; edges: few enough that the groups are fewer
@pytest.mark.parametrize("nl", [1, 2, 17, 64, 65, 255, 256, 257, 4095])
@pytest.mark.parametrize("m", [3000, 40000])
@pytest.mark.parametrize("hubs", [True, False])
def test_numbers_of_labels(ctx, nl, m, hubs):
    g = labelled(5000, m, nl, 40 + nl)
    if not hubs:
        ctx.set_hub_policy(64, 0)
    try:
        rg = ctx.upload(g)
    finally:
        ctx.set_hub_policy()
    for kind in (_lib.Q_WALK_HALF, _lib.Q_CYCLE):
        try:
            qs = G.queries(g, 2, 3, 4, kind, 5, 10 ** 6)
        except _lib.GpsmError:
            continue
        for i, q in enumerate(qs):
            check(rg, g, q, (kind, i))


@pytest.mark.parametrize("n", [2, 255, 256, 257, 1000])
def test_labels_in_blocks(ctx, n):
    """Each label's vertices next to each other in either order, with the
    sizes of vertex ranges: a path through all of them, forward and reversed."""
    for order in (1, -1):
        lab = (np.arange(n) * 4 // n + 1)[::order]
        g = G.from_edges(n, np.arange(n - 1), np.arange(1, n), lab)
        rg = ctx.upload(g)
        re = ctx.upload_edges(n, np.arange(n - 1), np.arange(1, n), lab)
        assert np.array_equal(re.g.row_offset, g.row_offset) and np.array_equal(re.g.col, g.col)
        for l in ([1, 1], [1, 2], [2, 1, 1], [4, 3], [2, 2, 3]):
            q = G.Query(np.array(l, dtype=np.uint32), np.arange(len(l) - 1, dtype=np.uint32),
                        np.arange(1, len(l), dtype=np.uint32))
            if set(l) <= set(lab.tolist()):
                check(rg, g, q, (order, l))
                check(re, g, q, (order, l))


def test_no_edges(ctx):
    g = G.from_edges(300, [], [], np.arange(300) % 5 + 1)
    q = G.Query(np.array([1, 2], dtype=np.uint32), np.array([0], dtype=np.uint32), np.array([1], dtype=np.uint32))
    assert ctx.upload(g).match(q).count == 0
    assert ctx.upload_edges(300, [], [], np.arange(300) % 5 + 1).match(q).count == 0


# 1024 entries a wave: a path's 2 (m - 1) just below, at and above, behind and
# before vertices without entries, and a star whose hub's fill several waves
@pytest.mark.parametrize("m", [512, 513, 514, 1025, 1537])
@pytest.mark.parametrize("gap", [0, 70])
def test_entry_blocks(ctx, m, gap):
    n = m + 2 * gap
    lab = np.arange(n) % 3 + 1
    v = np.arange(gap, gap + m)
    for src, dst in ((v[:-1], v[1:]), (np.full(m - 1, gap), v[1:])):
        g = G.from_edges(n, src, dst, lab)
        rg, re = ctx.upload(g), ctx.upload_edges(n, src, dst, lab)
        assert np.array_equal(re.g.row_offset, g.row_offset) and np.array_equal(re.g.col, g.col)
        for l in ([1, 2], [2, 1, 3], [3, 1, 3]):
            q = G.Query(np.array(l, dtype=np.uint32), np.arange(len(l) - 1, dtype=np.uint32),
                        np.arange(1, len(l), dtype=np.uint32))
            check(rg, g, q, l)
            check(re, g, q, l)
    bad = g.col.copy()
    bad[-1] = n
    with pytest.raises(_lib.GpsmError):
        ctx.upload(G.DataGraph(g.row_offset, bad, g.labels))
