"""Breadth-first join on a device with little memory left: smaller level
buffers, and plans handed to the depth-first join when even those do not fit."""
import ctypes as C

import pytest

from gpsm_amd import graphs as G
from gpsm_amd.matcher import Context
from test_zz_no_alloc import hip  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

MB = 1 << 20


class Ballast:
    """Device memory held until only `left` bytes are free."""

    def __init__(self, rt, left):
        self.rt, self.held = rt, []
        rt.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t)] * 2
        for chunk in (16 << 30, 1 << 30, 64 * MB):
            while self.free() >= left + chunk:
                p = C.c_void_p()
                if rt.hipMalloc(C.byref(p), chunk):
                    break
                self.held.append(p)

    def free(self):
        a, b = C.c_size_t(), C.c_size_t()
        assert self.rt.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    def drop(self):
        for p in self.held:
            self.rt.hipFree(p)


def fields(r):
    return (r.status, r.count, r.hash, r.level_rows, r.level_work, r.join_work, r.order)


# rows of levels 1 and 2 of a 4-cycle on 200k vertices: 1.2 GB at first, half a
# GB of it halved away; a triangle's first table of 16M rows: 1.3 GB, all of it
# needed
@pytest.mark.parametrize("n,m,k,left", [(200_000, 1_600_000, 4, 900), (1_000_000, 8_000_000, 3, 800)])
def test_little_memory(hip, n, m, k, left):  # noqa: F811
    g = G.small_graph(5, n=n, m=m, labels=1)
    qs = [G.cycle_query(k)]
    with Context(0) as ctx:
        rg = ctx.upload(g)
        ctx.profile(2)  # depth-first, and every other buffer at its size
        want = [fields(r) for r in rg.match_batch(qs)]
        ctx.profile(0)
        ballast = Ballast(hip, left * MB)
        try:
            assert ballast.free() < (left + 64) * MB
            got = [fields(r) for r in rg.match_batch(qs)]
        finally:
            ballast.drop()
        assert got == want and want[0][1] > 0
        assert [fields(r) for r in rg.match_batch(qs)] == want  # with all of the memory again
