"""The filter's and the candidate-edge tables' counted bytes (profile mode 2)
on cycles, where every count is known: n vertices of one label and degree 2,
all of them candidates of every vertex of a path of four."""
import pytest

from gpsm_amd import graphs as G

pytestmark = pytest.mark.gpu


def counted(ctx, rg, q, order):
    ctx.profile(2)
    try:
        r = rg.match_batch([q], explicit_orders=[order])[0]
        return r, {k: v["bytes"] for k, v in ctx.kernel_stats().items()}
    finally:
        ctx.profile(0)


@pytest.mark.parametrize("n", [64, 1000, 4099])
def test_path_on_a_cycle(ctx, n):
    r, b = counted(ctx, ctx.upload(G.cycle(n)), G.path_query(4), [0, 1, 2, 3])
    assert (r.status, r.count) == (0, 2 * n)
    W = (n + 31) // 32
    # ten supersteps' bitmap words: 1 explores 0 and 2, 2 explores 3, four
    # rounds refine 1 and 2.  Per neighbour explored n piece bounds and 2n keys,
    # then the fill: n vertex keys, n bounds, 2n entries and probes, n bits set.
    # Only the first round runs (it removes nothing): twice n bounds, 2n entries
    # and probes.
    explore, fill, refine = 8 * n + 4 * 2 * n, 4 * n + 8 * n + 4 * 2 * n + (2 * n + n) / 8, 8 * n + 4 * 2 * n + 2 * n / 8
    assert b["filter_step"] == 10 * 4 * W + 3 * (explore + fill) + 2 * refine
    # three forward tables: id, bounds and count of n candidates, 2n entries and probes
    assert b["cet_count"] == 3 * (16 * n + 4 * 2 * n + 2 * n / 8)
    # two tables written, the last one's sums, the records of the one before
    # (w's parent is y: a rank and a record per list entry)
    write = 16 * n + 4 * 2 * n + 2 * n / 8 + 4 * 2 * n
    sums = (12 + 32) * n + 4 * 2 * n + 2 * n / 8
    aggs = (8 + 32) * n + 2 * n * (4 + 8 + 32)
    assert b["cet_write"] == 2 * write + sums + aggs


def test_star_on_a_complete_graph(ctx):
    """0 - 1, 0 - 2, 0 - 3 from vertex 1: the first table runs against its edge
    and is counted again; the last two share a parent and a label, so their
    list entries are probed."""
    n = 40
    d = n - 1
    r, b = counted(ctx, ctx.upload(G.complete(n)), G.star_query(3), [1, 0, 2, 3])
    assert (r.status, r.count) == (0, n * d * (d - 1) * (d - 2))
    count = 16 * n + 4 * d * n + d * n / 8
    assert b["cet_count"] == 4 * count  # three forward, one again
    write = count + 4 * d * n
    sums = (12 + 32) * n + 4 * d * n + d * n / 8
    aggs = (8 + 32) * n + d * n * (4 + 1 / 8)
    assert b["cet_write"] == 2 * write + sums + aggs
