"""Arcs without a reverse arc: a vertex that only has arcs towards it joins no
community, but others join its own, so a coarse row has one member more than
arcs.  Communities around the sizes of the coarsening's wavefront (64 members)
and workgroup (1,024 arcs) rows, against numpy and the oracle.  Weights are
multiples of 2^-10: every sum is exact and must be equal."""
import numpy as np
import pytest

from parity import assert_runs_equal, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


def _csr(nv, rows, cols, seed):
    w = np.random.default_rng(seed).integers(1, 1024, len(rows)) / 1024.0
    order = np.lexsort((cols, rows))
    off = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=nv))]).astype(np.int64)
    return off, cols[order].astype(np.int64), w


def _sinks(sources, sink, stars=20):
    """Stars of `sources` vertices with one arc each into a sink without any.
    The sources of the stars take turns, so a source's next arc is another
    star's; the last source ends the CSR."""
    n = sources * stars
    src = np.arange(n) + (stars if sink == "first" else 0)
    return _csr(n + stars, src, np.arange(n) % stars + (0 if sink == "first" else n), n)


def _one_way(nv, seed):
    """0 to 3 arcs a vertex, most of them towards a few of them, mostly one-way."""
    rng = np.random.default_rng(seed)
    rows = np.repeat(np.arange(nv), rng.integers(0, 4, nv))
    cols = np.where(rng.random(len(rows)) < 0.7, rng.integers(nv // 60, size=len(rows)) * 60, rng.integers(nv, size=len(rows)))
    return _csr(nv, rows, cols, seed)


def _check_coarse(off, col, w, nb):
    import nido_amd as na
    g = na.GraphGPU((off, col, w), nb)
    g.singleton_partition()
    q = g.compute_modularity()
    for _ in range(2):
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
    return np.bincount(cid).max()


@pytest.mark.parametrize("sink", ["first", "last"])
@pytest.mark.parametrize("sources", [63, 64, 65, 255, 256, 1024, 1025])
def test_sinks(sources, sink):
    off, col, w = _sinks(sources, sink)
    print(f"case: stars of {sources} sources, sink {sink}", flush=True)
    assert _check_coarse(off, col, w, 2) == sources + 1
    assert_runs_equal(run_oracle(off, col, w, 2), run_gpu(off, col, w, 2))


def test_sinks_in_one_handle():
    import nido_amd as na
    graphs = [_sinks(n, s, 5) for n in (63, 64, 65, 130) for s in ("first", "last")]
    print("case: eight graphs of sinks in one handle", flush=True)
    b = na.BatchGPU(graphs, 2)
    b.run()
    for i, g in enumerate(graphs):
        assert np.array_equal(b.clustering(i), run_oracle(*g, 2)["clustering"])
    b.close()


@pytest.mark.parametrize("nv,nb", [(3000, 2), (40000, 8)])
def test_one_way_graph(nv, nb):
    off, col, w = _one_way(nv, nv)
    print(f"case: {nv} vertices, {len(col)} one-way arcs", flush=True)
    _check_coarse(off, col, w, nb)
    assert_runs_equal(run_oracle(off, col, w, nb), run_gpu(off, col, w, nb))
