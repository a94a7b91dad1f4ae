"""nido_modularity_noalloc at the edges of its arc tiles (2,048 arcs, 8 per
thread, 512 rows at a time): rows that cross tiles, empty rows between and
after them, offsets that do not start at 0.  The expected value is the
defining formula in integers: weights are multiples of 2^-10, so every sum is
exact and the comparison is for equality."""
from fractions import Fraction

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _expected(off, col, w, comm):
    src = np.repeat(np.arange(len(off) - 1), np.diff(off))
    c, x = col[off[0]:off[-1]], w[off[0]:off[-1]]
    twom = float(x.sum())
    if twom == 0.0:
        return 0.0
    inner = float(x[comm[src] == comm[c]].sum())
    totals = np.bincount(comm[src], weights=x, minlength=len(off) - 1) / twom
    terms = sum(round(Fraction(t * t) * 2 ** 64) for t in totals.tolist())
    return inner / twom - float(Fraction(terms, 2 ** 64))


@pytest.mark.parametrize("degrees,base", [
    ([1], 0),
    ([7, 8, 9, 0, 0, 1], 0),
    ([2047, 1, 2048, 2049], 0),
    ([0] * 600 + [5000] + [0] * 1100 + [3] + [0] * 700, 0),     # empty rows before, between and after
    ([1] * 4500, 3),                                            # more rows in a tile than are held at once
    ([14] * 3000 + [9000], 1),
])
def test_noalloc_at_tile_edges(degrees, base):
    import ctypes
    import nido_amd as na
    from test_zz_no_alloc import _setup
    _, hip = _setup()    # the library's own HIP runtime: another one cannot start after it in this process
    rng = np.random.default_rng(len(degrees) + base)
    nv, ne = len(degrees), sum(degrees)
    off = (base + np.concatenate([[0], np.cumsum(degrees)])).astype(np.int64)
    col = rng.integers(nv, size=base + ne)
    w = rng.integers(1, 2048, base + ne) / 1024.0
    comm = rng.integers(max(1, nv // 3), size=nv)
    bad = col.copy()
    bad[base + ne - 1] = nv
    print(f"case: {nv} rows, {ne} arcs from {base}", flush=True)
    dev, got = [], np.zeros(1)
    try:
        for x in (off, col, w, comm, bad, got):
            p = ctypes.c_void_p()
            assert hip.hipMalloc(ctypes.byref(p), x.nbytes) == 0
            dev.append(p.value)
            assert hip.hipMemcpy(p.value, x.ctypes.data, x.nbytes, 1) == 0
        assert hip.hipDeviceSynchronize() == 0
        d_off, d_col, d_w, d_comm, d_bad, d_q = dev

        def q(cols):
            na.modularity_noalloc(nv, base + ne, d_off, cols, d_w, d_comm, d_q, 0)
            assert hip.hipDeviceSynchronize() == 0
            assert hip.hipMemcpy(got.ctypes.data, d_q, 8, 2) == 0
            return float(got[0])
        expected = _expected(off, col, w, comm)
        for _ in range(2):                                      # the second call finds the first one's sums
            assert q(d_col) == expected
        assert np.isnan(q(d_bad))                               # an id out of range: NaN, and only for this call
        assert q(d_col) == expected
    finally:
        for p in dev:
            hip.hipFree(p)
