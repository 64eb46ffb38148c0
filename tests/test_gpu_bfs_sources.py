"""Breadth-first join with the learned order, whose rows take their candidates
from a back edge's vertex where that has fewer neighbours than the parent's
list: rows and work per level, budgets, levels that outgrow their buffer, all
as the depth-first join gives them, which reads the parents' lists only."""
import os

import numpy as np
import pytest

import pyoracle as O
from gpsm_amd import _lib, planner
from gpsm_amd import graphs as G
from test_gpu_bfs import depth_first, fields

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not os.path.exists(planner.WEIGHTS), reason="no trained planner weights")]
LEARNED = dict(order_mode=_lib.ORDER_LEARNED)


@pytest.fixture(scope="module")
def pctx(ctx):
    assert planner.install(ctx)
    return ctx


@pytest.mark.parametrize("hubs", [(8, 1 << 30), (512, 0)])
@pytest.mark.parametrize("labels", [1, 3])
def test_equals_depth_first_and_enumerator(pctx, labels, hubs):
    g = G.small_graph(80 + labels, n=1200, m=7000, labels=labels, kind="cl")
    qs = []
    for kind, kmax in ((_lib.Q_CYCLE, 5), (_lib.Q_CLIQUE, 5), (_lib.Q_WALK_INDUCED, 6)):
        qs += G.queries(g, 8, 3, kmax, kind, 19, 10 ** 6)
    try:
        pctx.set_hub_policy(*hubs)
        rg = pctx.upload(g)
    finally:
        pctx.set_hub_policy()
    got = [fields(r) for r in rg.match_batch(qs, **LEARNED)]
    assert got == depth_first(pctx, rg, qs, **LEARNED)
    for q, x in zip(qs, got):
        r1 = O.o1_enumerate(g, q)
        assert x[1:3] == (r1["count"], r1["hash"])


def two_uneven_bipartite(sizes, seed):
    """Per (left, right, edges): a bipartite graph whose left vertices have
    from very few to most of the right ones as neighbours, labels 2c + 1 and
    2c + 2."""
    rng = np.random.default_rng(seed)
    src, dst, labels, at = [], [], [], 0
    for c, (left, right, edges) in enumerate(sizes):
        w = 1.0 / np.arange(1, left + 1)
        src.append(at + rng.choice(left, edges, p=w / w.sum()))
        dst.append(at + left + rng.integers(0, right, edges))
        labels += [2 * c + 1] * left + [2 * c + 2] * right
        at += left + right
    return G.from_edges(at, np.concatenate(src), np.concatenate(dst), np.array(labels))


def labelled_cycle(a, b):
    return G.Query(np.array([a, b, a, b], dtype=np.uint32), np.array([0, 1, 2, 0], dtype=np.uint32),
                   np.array([1, 2, 3, 3], dtype=np.uint32))


def test_levels_outgrow_their_buffer_within_and_past_a_budget(pctx):
    """32 four-cycles on uneven bipartite graphs, 3e7 or more rows of the second level;
    then a budget that the wider graph's queries pass."""
    rg = pctx.upload(two_uneven_bipartite([(400, 2000, 90000), (200, 1000, 20000)], 3))
    qs = [labelled_cycle(1, 2), labelled_cycle(3, 4)] * 16
    base = [fields(r) for r in rg.match_batch(qs, **LEARNED)]
    assert sum(x[3][2] for x in base) > 1.5 * 2 ** 24
    assert base == depth_first(pctx, rg, qs, **LEARNED)
    assert base[:2] * 16 == base
    for budget in (base[1][5], base[0][5] - 1, base[0][5]):
        res = [fields(r) for r in rg.match_batch(qs, work_budget=budget, **LEARNED)]
        for x, b in zip(res, base):
            if b[5] <= budget:
                assert x == b
            else:
                assert x[:3] == (_lib.EBUDGET, 0, 0)


def test_budget_is_exact(pctx):
    g = G.small_graph(86, n=2000, m=16000, labels=2, kind="cl")
    rg = pctx.upload(g)
    qs = G.queries(g, 12, 4, 5, _lib.Q_CLIQUE, 31, 0) + G.queries(g, 12, 4, 4, _lib.Q_CYCLE, 32, 0)
    base = rg.match_batch(qs, **LEARNED)
    budget = sorted(r.join_work for r in base)[len(qs) // 2]
    for b in (budget, budget - 1):
        for r, r0 in zip(rg.match_batch(qs, work_budget=b, **LEARNED), base):
            want = (0, r0.count, r0.hash) if r0.join_work <= b else (_lib.EBUDGET, 0, 0)
            assert (r.status, r.count, r.hash) == want
