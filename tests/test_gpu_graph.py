"""A resident graph's derived arrays, built on the device: label statistics
on both sides of the histogram's width, rejected rows at wave edges, memory
reused by later graphs."""
import numpy as np
import pytest

import pyoracle as O
from gpsm_amd import _lib
from gpsm_amd import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("top", [3, 4095, 4096, 2 ** 32 - 1])
def test_label_values(ctx, top):
    """Labels up to and past the device histogram's 4096 entries."""
    g = G.small_graph(81, n=500, m=2500, labels=3, kind="cl")
    g.labels = np.where(g.labels == 3, np.uint32(top), g.labels)
    qs = G.queries(g, 6, 3, 5, _lib.Q_WALK_HALF, 9, 10 ** 6) if top < 10 ** 6 else [
        G.Query(np.array([top, 1, 2], dtype=np.uint32), np.array([0, 1], dtype=np.uint32),
                np.array([1, 2], dtype=np.uint32))]
    rg = ctx.upload(g)
    for q in qs:
        r = O.o1_enumerate(g, q)
        m = rg.match(q)
        assert (m.count, m.hash) == (r["count"], r["hash"])


@pytest.mark.parametrize("n", [2, 64, 65, 1024, 1025, 5000])
def test_vertex_ranges_and_hubs(ctx, n):
    """Sizes around a wave, a range block and a hub of more entries than a
    range holds: a star's closed forms."""
    g = G.from_edges(n, np.zeros(n - 1), np.arange(1, n), np.ones(n))
    rg = ctx.upload(g)
    re = ctx.upload_edges(n, np.zeros(n - 1), np.arange(1, n), np.ones(n))
    assert np.array_equal(re.g.row_offset, g.row_offset) and np.array_equal(re.g.col, g.col)
    for x in (rg, re):
        assert x.match(G.path_query(2)).count == 2 * (n - 1)
        if n > 2:
            assert x.match(G.path_query(3)).count == (n - 1) * (n - 2)
        assert x.hubs() == ((1, 64) if n - 1 > 64 else (0, 0))


@pytest.mark.parametrize("row", [0, 63, 64, 199])
def test_bad_rows_are_rejected(ctx, row):
    g = G.cycle(200)
    lo = int(g.row_offset[row])
    for change in ("swap", "duplicate", "self", "range"):
        col = g.col.copy()
        if change == "swap":
            col[lo], col[lo + 1] = col[lo + 1], col[lo]
        elif change == "duplicate":
            col[lo + 1] = col[lo]
        elif change == "self":
            col[lo] = row
        else:
            col[lo + 1] = 200
        with pytest.raises(_lib.GpsmError) as e:
            ctx.upload(G.DataGraph(g.row_offset, col, g.labels))
        assert e.value.code == -1
    labels = g.labels.copy()
    labels[row] = 0
    with pytest.raises(_lib.GpsmError) as e:
        ctx.upload(G.DataGraph(g.row_offset, g.col, labels))
    assert e.value.code == -1
    assert ctx.upload(g).match(G.path_query(3)).count == 400


def test_graphs_reuse_memory(ctx):
    """Graphs of changing sizes made and freed in turn, one kept throughout."""
    specs = [(400, 1600), (3000, 12000), (401, 1601), (3000, 12001), (50, 100)]
    graphs = [G.small_graph(90 + i, n=n, m=m, labels=2, kind="cl") for i, (n, m) in enumerate(specs)]
    q = G.path_query(3)
    kept = ctx.upload(graphs[1])
    want = [ctx.upload(g).match(q) for g in graphs]
    for rep in range(3):
        for g, w in zip(graphs, want):
            src, dst = g.edges()
            for rg in (ctx.upload(g), ctx.upload_edges(g.n, src, dst, g.labels)):
                r = rg.match(q)
                assert (r.count, r.hash) == (w.count, w.hash)
                rg.free()
    assert kept.match(q).hash == want[1].hash
