"""Allocation-free scans of several contexts at the same time: they share one
scratch array per device."""
import threading

import numpy as np
import pytest

from gpsm_amd.matcher import Context
from test_zz_no_alloc import DevArray, hip, noalloc_scan  # noqa: F401  (hip: fixture)

pytestmark = pytest.mark.gpu


def test_overlapping_calls_take_turns(hip):  # noqa: F811
    """Four threads, a context each, sizes of one, a few and many tiles, so
    that every call clears states which the others' lengths would still need."""
    sizes = (5_000_003, 32_768, 40_000_000, 1_000_001)
    calls = 12
    got, errors = [[] for _ in sizes], []

    def work(i):
        try:
            rng = np.random.default_rng(i)
            a = rng.integers(0, 1 << 32, size=sizes[i], dtype=np.uint64)
            want = np.zeros(len(a), dtype=np.uint64)
            np.cumsum(a[:-1], out=want[1:])
            with Context(0) as c:
                din, dout = DevArray(hip, len(a)), DevArray(hip, len(a))
                din.put(a.astype(np.uint32))
                start.wait(60)
                for _ in range(calls):
                    got[i].append(noalloc_scan(c, din.p, dout.p, len(a)) == (0, int(a.sum()))
                                  and np.array_equal(dout.get(), want.astype(np.uint32)))
                din.free()
                dout.free()
        except Exception as e:  # noqa: BLE001
            errors.append(e)
            start.abort()

    start = threading.Barrier(len(sizes))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(100)
    assert not errors and not any(t.is_alive() for t in threads)
    assert got == [[True] * calls] * len(sizes)
