"""Tiles of 2,048 arcs that span few and very many rows, most of them empty:
vertex weights and whole runs against numpy and the oracle, and the
allocation-free modularity against the handle's.  Weights are multiples of
2^-10, so every sum is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _spread(rows, gap, hub, seed):
    """`rows` vertices with arcs, `gap` empty ones after each, a hub joined to
    all of them in front when `hub` is set, otherwise a ring; symmetric."""
    rng = np.random.default_rng(seed)
    nv = rows * (gap + 1) + 1
    at = 1 + np.arange(rows) * (gap + 1)
    other = np.zeros(rows, dtype=np.int64) if hub else np.roll(at, -1)
    u, v = np.concatenate([at, rng.choice(at, rows)]), np.concatenate([other, rng.choice(at, rows)])
    key = np.unique(np.minimum(u, v)[u != v] * nv + np.maximum(u, v)[u != v])
    lo, hi = key // nv, key % nv
    w = rng.integers(1, 2048, len(key)) / 1024.0
    r, c, ww = np.concatenate([lo, hi]), np.concatenate([hi, lo]), np.concatenate([w, w])
    order = np.lexsort((c, r))
    off = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=nv))]).astype(np.int64)
    return off, c[order].astype(np.int64), ww[order]


@pytest.mark.parametrize("rows,gap,hub", [
    (3, 5000, False),          # one short tile over more than 8,192 rows
    (600, 7, False),           # about 4,096 rows a tile
    (1500, 1, True),
    (4000, 60, True),          # tiles that start in the hub's row and end far after it
    (900, 400, False),
])
def test_rows_far_apart(rows, gap, hub):
    import ctypes
    import nido_amd as na
    from parity import assert_runs_equal, run_gpu, run_oracle
    from test_zz_no_alloc import _setup
    _, hip = _setup()
    off, col, w = _spread(rows, gap, hub, rows + gap)
    nv = len(off) - 1
    print(f"case: {rows} rows, {gap} empty after each, {len(col)} arcs", flush=True)
    k = np.bincount(np.repeat(np.arange(nv), np.diff(off)), weights=w, minlength=nv)
    g = na.GraphGPU((off, col, w), 2)
    assert np.array_equal(g.vertex_weights(), k)
    g.singleton_partition()
    q = g.compute_modularity()
    g.louvain_iteration(q)
    comm, expected = g.communities(), g.compute_modularity()
    g.close()
    dev, got = [], np.zeros(1)
    try:
        for x in (off, col, w, comm, got):
            p = ctypes.c_void_p()
            assert hip.hipMalloc(ctypes.byref(p), x.nbytes) == 0
            dev.append(p.value)
            assert hip.hipMemcpy(p.value, x.ctypes.data, x.nbytes, 1) == 0
        na.modularity_noalloc(nv, len(col), *dev[:4], dev[4], 0)
        assert hip.hipDeviceSynchronize() == 0
        assert hip.hipMemcpy(got.ctypes.data, dev[4], 8, 2) == 0
    finally:
        for p in dev:
            hip.hipFree(p)
    assert got[0] == expected
    assert_runs_equal(run_oracle(off, col, w, 2), run_gpu(off, col, w, 2))
