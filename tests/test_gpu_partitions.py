"""Whole runs against the oracle on graphs whose long rows sit at the edges of
a split into partitions: one, two and three or more of them, rows that just
fit the key limit, and counts of partitions that are no power of two."""
import numpy as np
import pytest

from parity import assert_runs_equal, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


def _hubs(degrees, n, seed):
    """A hub per degree, joined to that many of n other vertices, and n weak
    edges between those."""
    rng = np.random.default_rng(seed)
    h = len(degrees)
    u = np.concatenate([np.full(d, i) for i, d in enumerate(degrees)] + [h + rng.integers(n, size=n)])
    v = np.concatenate([h + rng.permutation(n)[:d] for d in degrees] + [h + rng.integers(n, size=n)])
    nv = h + n
    key = np.unique(np.minimum(u, v) * nv + np.maximum(u, v))
    lo, hi = key // nv, key % nv
    lo, hi = lo[lo != hi], hi[lo != hi]
    w = 1.0 - rng.random(len(lo))
    order = np.lexsort((np.concatenate([hi, lo]), np.concatenate([lo, hi])))
    rows, cols = np.concatenate([lo, hi])[order], np.concatenate([hi, lo])[order]
    off = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=nv))]).astype(np.int64)
    return off, cols.astype(np.int64), np.concatenate([w, w])[order]


@pytest.mark.parametrize("degrees,n,knobs", [
    ([875, 876, 877, 1023, 1024, 1025], 3000, {}),
    ([1751, 1752, 1753, 2047, 2048, 2049, 2628, 2629], 6000, {}),
    ([4096, 8191, 8192, 8193, 11000], 12000, {}),
    ([40, 41, 64, 65, 100, 128, 129, 2000], 3000, {"big_min_deg": 32, "big_part_arcs": 64, "big_key_limit": 64}),
    ([600, 1300, 3000], 4000, {"big_part_arcs": 1025}),       # above the limit: rows through the HBM table
])
def test_partitioned_rows_match_the_oracle(degrees, n, knobs):
    off, col, w = _hubs(degrees, n, len(degrees) * n)
    print(f"case: hubs of {degrees}, {knobs}", flush=True)
    assert list(np.diff(off)[:len(degrees)]) == degrees
    assert_runs_equal(run_oracle(off, col, w, 4), run_gpu(off, col, w, 4, **knobs))
