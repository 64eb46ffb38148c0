"""The breadth-first join of plans with back edges against the depth-first
one (which a batch whose join bytes are counted runs), the enumerator and
closed forms: short and long candidate lists, lists taken from a back edge's
adjacency, levels that outgrow their buffer, more plans than one launch
holds, budgets."""
import numpy as np
import pytest

import pyoracle as O
from gpsm_amd import _lib
from gpsm_amd import graphs as G

pytestmark = pytest.mark.gpu


def fields(r):
    return (r.status, r.count, r.hash, r.level_rows, r.level_work, r.join_work, r.order)


def depth_first(ctx, rg, qs, **kw):
    ctx.profile(2)
    try:
        return [fields(r) for r in rg.match_batch(qs, **kw)]
    finally:
        ctx.profile(0)


def two_hubs(leaves):
    """Two hubs, each adjacent to every leaf: 4-cycles alternate hub and leaf."""
    src = np.repeat(np.arange(2), leaves)
    dst = 2 + np.tile(np.arange(leaves), 2)
    return G.from_edges(2 + leaves, src, dst, np.ones(2 + leaves))


@pytest.mark.parametrize("hubs", [(8, 1 << 30), (512, 0)])
@pytest.mark.parametrize("labels", [1, 3])
def test_equals_depth_first_and_enumerator(ctx, labels, hubs):
    g = G.small_graph(70 + labels, n=1200, m=7000, labels=labels, kind="cl")
    qs = []
    for kind, kmax in ((_lib.Q_CYCLE, 5), (_lib.Q_CLIQUE, 5), (_lib.Q_WALK_INDUCED, 6)):
        qs += G.queries(g, 8, 3, kmax, kind, 17, 10 ** 6)
    try:
        ctx.set_hub_policy(*hubs)
        rg = ctx.upload(g)
    finally:
        ctx.set_hub_policy()
    got = [fields(r) for r in rg.match_batch(qs)]
    assert got == depth_first(ctx, rg, qs)
    for q, x in zip(qs, got):
        r1 = O.o1_enumerate(g, q)
        assert x[1:3] == (r1["count"], r1["hash"])


@pytest.mark.parametrize("leaves", [511, 512, 513, 700])
def test_long_lists(ctx, leaves):
    """Candidate lists just below, at and above the length a workgroup takes."""
    rg = ctx.upload(two_hubs(leaves))
    r = rg.match_batch([G.cycle_query(4)])[0]
    assert r.count == 4 * leaves * (leaves - 1)
    assert fields(r) == depth_first(ctx, rg, [G.cycle_query(4)])[0]


def test_level_outgrows_its_buffer(ctx):
    """1.8e7 rows of the second level where the mean fan-out suggests 1e4."""
    rg = ctx.upload(two_hubs(3000))
    qs = [G.cycle_query(4), G.path_query(4), G.clique_query(3)]
    res = rg.match_batch(qs)
    assert res[0].count == 4 * 3000 * 2999 and res[2].count == 0
    assert res[0].level_rows[2] > 10 ** 7
    assert [fields(r) for r in res] == depth_first(ctx, rg, qs)


def test_more_plans_than_a_launch_holds(ctx):
    g = G.small_graph(75, n=800, m=5000, labels=2, kind="cl")
    rg = ctx.upload(g)
    qs = G.queries(g, 20, 3, 4, _lib.Q_CLIQUE, 5, 0) * 27  # 540
    res = [fields(r) for r in rg.match_batch(qs)]
    assert res == depth_first(ctx, rg, qs)
    assert res[:20] == res[-20:] == [fields(r) for r in rg.match_batch(qs[:20])]


def test_budget_is_exact(ctx):
    g = G.small_graph(76, n=2000, m=16000, labels=2, kind="cl")
    rg = ctx.upload(g)
    qs = G.queries(g, 12, 4, 5, _lib.Q_CLIQUE, 29, 0) + G.queries(g, 12, 4, 4, _lib.Q_CYCLE, 30, 0)
    base = rg.match_batch(qs)
    budget = sorted(r.join_work for r in base)[len(qs) // 2]
    for b in (budget, budget - 1):
        for r, r0 in zip(rg.match_batch(qs, work_budget=b), base):
            want = (0, r0.count, r0.hash) if r0.join_work <= b else (_lib.EBUDGET, 0, 0)
            assert (r.status, r.count, r.hash) == want
