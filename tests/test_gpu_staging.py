"""Large copies through the context's staging (4 MB halves, from 1 MB on): a
CSR to the device and back, and text cut off at a capacity, at sizes one word
around those."""
import ctypes as C

import numpy as np
import pytest

from gpsm_amd import _lib
from gpsm_amd import graphs as G

pytestmark = pytest.mark.gpu


# 8 bytes of columns per edge: one word below and above 1 MB, 4 MB, 8 MB, and three halves
@pytest.mark.parametrize("edges", [131071, 131072, 524287, 524288, 524289, 1048576, 1048577, 1572865])
def test_csr_round_trip(ctx, edges):
    r = np.random.default_rng(edges)
    n = edges + 1
    ids = r.permutation(n).astype(np.uint32)
    src, dst, lab = ids[:-1], ids[1:], r.integers(1, 5, n).astype(np.uint32)
    g = G.from_edges(n, src, dst, lab)
    rg = ctx.upload_edges(n, src, dst, lab)
    assert np.array_equal(rg.g.row_offset, g.row_offset) and np.array_equal(rg.g.col, g.col)
    # uploaded as a CSR: the same graph (edges counted per label pair)
    up = ctx.upload(g)
    ro, col = np.zeros(n + 1, dtype=np.uint32), np.zeros(2 * edges, dtype=np.uint32)
    _lib.check(_lib.lib().gpsm_graph_csr(up.h, _lib.ptr(ro), _lib.ptr(col)), "gpsm_graph_csr")
    assert np.array_equal(ro, g.row_offset) and np.array_equal(col, g.col)
    q = G.Query(np.array([1, 2], dtype=np.uint32), np.array([0], dtype=np.uint32), np.array([1], dtype=np.uint32))
    want = int((((lab[src] == 1) & (lab[dst] == 2)) | ((lab[src] == 2) & (lab[dst] == 1))).sum())
    assert up.match(q).count == rg.match(q).count == want


@pytest.mark.parametrize("cap", [0, 1, (1 << 20) - 1, 1 << 20, (4 << 20) + 1, (8 << 20) + 1, 16_000_000])
def test_text_capacity(ctx, cap):
    t = np.random.default_rng(3).integers(0, 10 ** 6, (400_000, 3)).astype(np.uint32)
    line = "".join("(%d, %d) " % (j, v) for j, v in enumerate(t[0])) + "\n"
    text, need = np.zeros(max(cap, 1), dtype=np.uint8), C.c_uint64()
    full, fneed = np.zeros(20_000_000, dtype=np.uint8), C.c_uint64()
    call = _lib.lib().gpsm_format_tuples
    assert call(ctx.h, _lib.ptr(t), len(t), 3, None, _lib.ptr(full), full.size, C.byref(fneed)) == 0
    rc = call(ctx.h, _lib.ptr(t), len(t), 3, None, _lib.ptr(text), cap, C.byref(need))
    assert need.value == fneed.value and rc == (0 if cap >= need.value else -5)
    assert bytes(full[:len(line)]) == line.encode()
    assert np.array_equal(text[:min(cap, need.value)], full[:min(cap, need.value)])
