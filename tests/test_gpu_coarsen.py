"""The coarse graph after an aggregation against numpy on the same
communities: coarse rows at the edges of the wavefront (64 arcs), workgroup
(1,024 arcs) and HBM-table aggregation, and of the 4,096-arc tiles the latter
insert.  Weights are multiples of 2^-10, so every sum is exact in FP64 and
the coarse weights must be equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _stars(leaves, links, seed):
    """Stars with the given numbers of leaves, their centres in a ring and
    `links` more weak edges between random vertices."""
    rng = np.random.default_rng(seed)
    start = np.concatenate([[0], np.cumsum([n + 1 for n in leaves])])
    nv = int(start[-1])
    u = np.concatenate([np.full(n, s) for n, s in zip(leaves, start)] + [start[:-1], rng.integers(nv, size=links)])
    v = np.concatenate([np.arange(s + 1, s + 1 + n) for n, s in zip(leaves, start)] +
                       [np.roll(start[:-1], -1), rng.integers(nv, size=links)])
    w = np.concatenate([rng.integers(512, 1025, sum(leaves)), rng.integers(1, 8, len(leaves) + links)]) / 1024.0
    key, at = np.unique(np.minimum(u, v) * nv + np.maximum(u, v), return_index=True)
    lo, hi, w = key // nv, key % nv, w[at]
    loop = lo == hi                                  # a self arc is one arc
    rows, cols = np.concatenate([lo, hi[~loop]]), np.concatenate([hi, lo[~loop]])
    ws = np.concatenate([w, w[~loop]])
    order = np.lexsort((cols, rows))
    off = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=nv))]).astype(np.int64)
    return off, cols[order].astype(np.int64), ws[order]


@pytest.mark.parametrize("leaves,links", [
    ([1, 1, 2, 30, 31, 32, 33], 0),                              # rows of 4 to 68 arcs
    ([30, 31, 32, 33, 500, 510, 511, 512, 513], 200),            # around 64 and 1,024 arcs
    ([2046, 2047, 2048, 2049, 511, 512, 1, 1], 30),              # around one tile of 4,096 arcs
    ([20000, 3, 3, 700, 700, 9000] + [5] * 300, 3000),           # a community far above the others
    ([4] * 2000 + [6000] * 3, 20000),                            # HBM rows with many targets
])
def test_coarse_graph_equals_numpy(leaves, links):
    import nido_amd as na
    off, col, w = _stars(leaves, links, len(leaves))
    print(f"case: {len(leaves)} stars, {links} links, {len(col)} arcs", flush=True)
    g = na.GraphGPU((off, col, w), 32)   # with few batches a star's centre and leaves swap and nothing forms
    g.singleton_partition()
    q = g.compute_modularity()
    for _ in range(3):
        q, _, _ = g.louvain_iteration(q)
    comm = g.communities()
    assert not g.aggregation()
    noff, ncol, nw = g.graph()
    g.close()
    ids, cid = np.unique(comm, return_inverse=True)
    k = len(ids)
    assert len(noff) == k + 1
    key, at = np.unique(cid[np.repeat(np.arange(len(off) - 1), np.diff(off))] * k + cid[col], return_inverse=True)
    got = np.repeat(np.arange(k), np.diff(noff)) * k + ncol
    order = np.argsort(got)
    assert np.array_equal(got[order], key)
    assert np.array_equal(nw[order], np.bincount(at, weights=w))
