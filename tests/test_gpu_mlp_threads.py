"""A network of one context as the planner of another, called by that
context's thread while its own context's thread calls a second network."""
import threading

import numpy as np
import pytest

from gpsm_amd import _lib, planner
from gpsm_amd import graphs as G
from gpsm_amd.matcher import Context

pytestmark = pytest.mark.gpu


def test_planner_of_another_context(ctx):
    rng = np.random.default_rng(3)
    # sizes that make the staging grow while the other thread's calls use theirs
    xs = [rng.standard_normal((b, _lib.FEAT)).astype(np.float32) for b in (7, 300, 4000, 64, 9000, 30000)]
    ts = [rng.standard_normal(len(x)).astype(np.float32) for x in xs]
    own, lent = planner.MLP(ctx, seed=1), planner.MLP(ctx, seed=2)
    want = [own.forward(x) for x in xs]
    want_loss = [own.grad(x, t)[0] for x, t in zip(xs, ts)]
    g = G.small_graph(71, n=1200, m=7000, labels=3, kind="cl")
    qs = G.queries(g, 24, 4, 6, _lib.Q_WALK_INDUCED, 17, 10 ** 6)
    with Context(0) as other:
        rg = other.upload(g)
        _lib.check(_lib.lib().gpsm_set_planner(other.h, lent.h), "gpsm_set_planner")

        def batch():
            return [(r.status, r.count, r.hash, r.order) for r in rg.match_batch(qs, order_mode=_lib.ORDER_LEARNED)]

        want_batch = batch()
        got, errors, done = [], [], threading.Event()

        def matches():
            try:
                for _ in range(60):
                    got.append(batch() == want_batch)
            except Exception as e:  # noqa: BLE001
                errors.append(e)
            done.set()

        t = threading.Thread(target=matches)
        t.start()
        rounds = 0
        while not done.is_set() or rounds < 3:
            for x, tt, y, loss in zip(xs, ts, want, want_loss):
                assert np.array_equal(own.forward(x), y)
                # positive terms; up to 938 workgroups' sums added in any order,
                # twice 938 + 5 roundings of 2^-24
                assert abs(own.grad(x, tt)[0] - loss) <= 1.2e-4 * loss
            rounds += 1
        t.join(60)
        assert not errors and got == [True] * 60
        _lib.check(_lib.lib().gpsm_set_planner(other.h, None), "gpsm_set_planner")
    own.free()
    lent.free()


def test_network_freed_after_its_context():
    c = Context(0)
    m = planner.MLP(c, seed=1)
    y = m.forward(np.ones((40000, _lib.FEAT), dtype=np.float32))
    assert np.isfinite(y).all()
    c.close()
    m.free()
