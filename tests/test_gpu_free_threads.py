"""Graphs freed by another thread than the context's, whose batches capture
hipGraphs meanwhile."""
import threading

import pytest

from gpsm_amd import _lib
from gpsm_amd import graphs as G
from gpsm_amd.matcher import Context

pytestmark = pytest.mark.gpu


def test_graphs_freed_while_batches_are_captured():
    small = G.small_graph(21, n=300, m=900, labels=2)
    g = G.small_graph(22, n=4000, m=16000, labels=2)
    # batches of different numbers of queries: a capture for each
    sets = [G.queries(g, 1 + i, 4, 6, _lib.Q_WALK_TREE, 40 + i, 10 ** 6) for i in range(8)]
    with Context(0) as ctx:
        rg = ctx.upload(g)
        want = [[(r.status, r.count, r.hash) for r in rg.match_batch(qs)] for qs in sets]
        for _ in range(4):
            others = [ctx.upload(small) for _ in range(60)]
            ready = threading.Event()

            def drop():
                ready.wait(30)
                for x in others:
                    x.free()

            t = threading.Thread(target=drop)
            t.start()
            try:
                ready.set()
                while True:
                    alive = t.is_alive()
                    for qs, w in zip(sets, want):
                        assert [(r.status, r.count, r.hash) for r in rg.match_batch(qs, use_graph=True)] == w
                    if not alive:
                        break
            finally:
                t.join(30)


def test_context_closed_while_its_graphs_are_freed():
    small = G.small_graph(21, n=300, m=900, labels=2)
    for _ in range(3):
        ctx = Context(0)
        graphs = [ctx.upload(small) for _ in range(60)]
        t = threading.Thread(target=lambda: [x.free() for x in graphs])
        t.start()
        ctx.close()
        t.join(30)
        assert all(x.h is None for x in graphs)
