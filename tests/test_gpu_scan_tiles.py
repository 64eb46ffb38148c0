"""The one-pass scan at the edges of its tiles (32768 values, quads of four) and
of the 64 tiles looked back over at a time, on aligned and unaligned device
arrays, in place, with sums past 32 bits."""
import ctypes as C

import numpy as np
import pytest

from test_zz_no_alloc import DevArray, hip, noalloc_scan  # noqa: F401

pytestmark = pytest.mark.gpu
T = 32768


@pytest.mark.parametrize("n", [1, 3, 4, 5, 2047, 2048, T - 1, T, T + 1, 2 * T + 3, 63 * T, 64 * T, 64 * T + 1, 65 * T,
                               129 * T + 5])
def test_tiles(ctx, hip, n):  # noqa: F811
    a = np.random.default_rng(n).integers(0, 2 ** 32, n, dtype=np.uint32)
    want = np.zeros(n + 1, dtype=np.uint64)
    np.cumsum(a, dtype=np.uint64, out=want[1:])
    buf = DevArray(hip, 2 * (n + 8))
    for off_in, off_out, same in ((0, 0, False), (1, 0, False), (0, 3, False), (2, 2, True), (0, 0, True)):
        h = np.full(2 * (n + 8), 7, dtype=np.uint32)
        h[off_in:off_in + n] = a
        buf.put(h)
        at = off_in if same else n + 8 + off_out
        for _ in range(1 if same else 2):  # the scratch is used again
            rc, total = noalloc_scan(ctx, C.c_void_p(buf.p.value + 4 * off_in), C.c_void_p(buf.p.value + 4 * at), n)
            assert rc == 0 and total == int(want[-1]), (off_in, off_out)
        h[at:at + n] = want[:-1].astype(np.uint32)
        assert np.array_equal(buf.get(), h), (off_in, off_out)  # and nothing beside it
    buf.free()
