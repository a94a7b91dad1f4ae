"""Handles that take each other's freed device memory: graphs of neighbouring
and of very different sizes, created, run and closed over and over in several
threads, and one after another on one handle's memory across phases, against
the oracle."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ring(n, seed):
    """A ring of n vertices with n random chords, weights multiples of 2^-10."""
    rng = np.random.default_rng(seed)
    u = np.concatenate([np.arange(n), rng.integers(n, size=n)])
    v = np.concatenate([(np.arange(n) + 1) % n, rng.integers(n, size=n)])
    key = np.unique(np.minimum(u, v)[u != v] * n + np.maximum(u, v)[u != v])
    lo, hi = key // n, key % n
    w = rng.integers(1, 2048, len(key)) / 1024.0
    r, c, ww = np.concatenate([lo, hi]), np.concatenate([hi, lo]), np.concatenate([w, w])
    order = np.lexsort((c, r))
    off = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int64)
    return off, c[order].astype(np.int64), ww[order]


def test_handles_share_freed_memory():
    from parity import assert_runs_equal, run_gpu, run_oracle
    graphs = [_ring(n, n) for n in (3, 100, 107, 2000, 2047, 2300, 30000)]
    expected = [run_oracle(*g, 2) for g in graphs]
    errors = []

    def work(t):
        try:
            for i in range(14):
                k = (i * (2 * t + 1) + t) % len(graphs)
                assert_runs_equal(expected[k], run_gpu(*graphs[k], 2))
        except BaseException as e:   # noqa: BLE001 (handed to the test's thread)
            errors.append(e)
    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if errors:
        raise errors[0]
