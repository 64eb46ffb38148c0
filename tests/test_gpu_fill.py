"""The sets an explore step hands its neighbours, whichever way they are
filled: pulled by the neighbours' vertices, pushed by few candidates, pushed
by hubs in parts, pushed by the ops themselves in a wide batch."""
import numpy as np
import pytest

import pyoracle as O
from gpsm_amd import graphs as G

pytestmark = pytest.mark.gpu


def hub_graph(n, m, rare, seed):
    """Two hubs of more entries than a vertex range holds (4096), over a random
    graph; label 1 on the hubs and `rare` others, labels 2 and 3 on the rest."""
    r = np.random.default_rng(seed)
    hub = np.arange(2)
    a = np.concatenate([r.integers(0, n, m), np.repeat(hub, 4200)])
    b = np.concatenate([r.integers(0, n, m)] + [2 + r.choice(n - 2, 4200, replace=False) for _ in hub])
    keep = a != b
    labels = r.integers(2, 4, n)
    labels[:2] = 1
    labels[2 + r.choice(n - 2, rare, replace=False)] = 1
    e = np.unique(np.stack([np.minimum(a, b), np.maximum(a, b)], 1)[keep], axis=0)
    return G.from_edges(n, e[:, 0], e[:, 1], labels)


def star(labels):
    k = len(labels)
    return G.Query(np.array(labels, dtype=np.uint32), np.zeros(k - 1, dtype=np.uint32),
                   np.arange(1, k, dtype=np.uint32))


def caterpillar(labels):
    """A path of three with one leaf at each end and two in the middle."""
    return G.Query(np.array(labels, dtype=np.uint32), np.array([0, 1, 0, 1, 1, 2], dtype=np.uint32),
                   np.array([1, 2, 3, 4, 5, 6], dtype=np.uint32))


QUERIES = [star([1, 2]), star([2, 1]), star([1, 2, 3, 2]), star([2, 1, 3, 3]), star([3, 2, 2, 3, 1]),
           caterpillar([1, 2, 3, 2, 3, 1, 2]), caterpillar([2, 3, 2, 1, 3, 2, 3]), caterpillar([3, 2, 1, 2, 3, 2, 2])]


# rare: the rare label's vertices, from far below to far above 1/32 of a common one's
@pytest.mark.parametrize("rare", [0, 5, 130, 2000])
@pytest.mark.parametrize("m", [4000, 16000])
def test_fills_match_oracle(ctx, rare, m):
    g = hub_graph(9000, m, rare, 7 + rare)
    rg = ctx.upload(g)
    for i, q in enumerate(QUERIES):
        st, _, ref, _ = O.o2_filter(g, q)
        bm, cnt = rg.filter(q)
        if st != O.OK:
            assert (cnt == 0).any(), i
            continue
        for u in range(q.n):
            bits = np.unpackbits(bm[u].view(np.uint8), bitorder="little")[:g.n]
            assert np.array_equal(bits != 0, ref[u] != 0), (i, u)


def test_wide_batch_equals_single_queries(ctx):
    """150 queries on 2^20 vertices: more pairs of op and vertex range (at
    least 1024 ranges) than one launch visits unlisted, so the ops push."""
    g = hub_graph(1 << 20, 1 << 20, 3000, 11)
    rg = ctx.upload(g)
    one = [(r.cand, r.count, r.hash) for r in (rg.match(q) for q in QUERIES)]
    got = [(r.cand, r.count, r.hash) for r in rg.match_batch([QUERIES[i % len(QUERIES)] for i in range(150)])]
    for i, r in enumerate(got):
        a = one[i % len(QUERIES)]
        assert np.array_equal(r[0], a[0]) and r[1:] == a[1:], i
