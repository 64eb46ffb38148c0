"""Breadth-first levels that stop at a full buffer and go on later, when some
of the batch's queries have passed their work budget in between."""
import numpy as np
import pytest

from gpsm_amd import _lib
from gpsm_amd import graphs as G

pytestmark = pytest.mark.gpu


def two_pairs_of_hubs(a, b):
    """Two hubs (label 2) with a common leaves (label 1), two more (label 4)
    with b (label 3)."""
    src, dst, labels, at = [], [], [], 0
    for leaves, leaf, hub in ((a, 1, 2), (b, 3, 4)):
        src.append(at + np.repeat(np.arange(2), leaves))
        dst.append(at + 2 + np.tile(np.arange(leaves), 2))
        labels += [hub] * 2 + [leaf] * leaves
        at += 2 + leaves
    return G.from_edges(at, np.concatenate(src), np.concatenate(dst), np.array(labels))


def labelled_cycle(leaf, hub):
    return G.Query(np.array([leaf, hub, leaf, hub], dtype=np.uint32), np.array([0, 1, 2, 0], dtype=np.uint32),
                   np.array([1, 2, 3, 3], dtype=np.uint32))


@pytest.mark.parametrize("a,b", [(501, 201), (385, 129)])
def test_budget_passed_while_a_level_waits_for_its_buffer(ctx, a, b):
    """Two plans in turn, their rows in the same groups of four at every change
    of plan; their second levels together are several buffers long.  The wider
    plan's queries pass the budget while the level waits, the others' must
    come out whole."""
    wide, narrow = labelled_cycle(1, 2), labelled_cycle(3, 4)
    qs = [wide, narrow] * 128
    orders = [[0, 1, 2, 3]] * len(qs)
    rg = ctx.upload(two_pairs_of_hubs(a, b))
    base = rg.match_batch(qs, explicit_orders=orders)
    for r, leaves in zip(base, [a, b] * 128):
        assert (r.status, r.count, r.level_rows[2]) == (0, 2 * leaves * (leaves - 1), 2 * leaves * (leaves - 1))
    assert sum(r.level_rows[2] for r in base) > 1.2 * 2 ** 24
    # passed on the way through the second level, not before it
    w = base[0].level_work
    budget = w[1] + w[2] + w[3] // 10
    assert base[1].join_work < budget < base[0].join_work
    res = rg.match_batch(qs, explicit_orders=orders, work_budget=budget)
    for r, r0 in zip(res[1::2], base[1::2]):
        assert (r.status, r.count, r.hash, r.level_rows, r.level_work, r.join_work) == \
            (0, r0.count, r0.hash, r0.level_rows, r0.level_work, r0.join_work)
    for r in res[0::2]:
        assert (r.status, r.count, r.hash) == (_lib.EBUDGET, 0, 0)


@pytest.mark.parametrize("part", [16, 10, 6, 4, 3, 2])
def test_budget_passed_at_any_time(ctx, part):
    """The budget passed earlier or later on the way through the second level:
    rows are left out before a wave stops in a step as well as after."""
    wide, narrow = labelled_cycle(1, 2), labelled_cycle(3, 4)
    qs = [wide, narrow] * 128
    orders = [[0, 1, 2, 3]] * len(qs)
    rg = ctx.upload(two_pairs_of_hubs(501, 201))
    base = rg.match_batch(qs, explicit_orders=orders)
    w = base[0].level_work
    budget = w[1] + w[2] + w[3] // part
    assert base[1].join_work < budget < base[0].join_work
    for _ in range(5):
        res = rg.match_batch(qs, explicit_orders=orders, work_budget=budget)
        for r, r0 in zip(res[1::2], base[1::2]):
            assert (r.status, r.count, r.hash, r.level_rows, r.level_work, r.join_work) == \
                (0, r0.count, r0.hash, r0.level_rows, r0.level_work, r0.join_work)
        for r in res[0::2]:
            assert (r.status, r.count, r.hash) == (_lib.EBUDGET, 0, 0)
