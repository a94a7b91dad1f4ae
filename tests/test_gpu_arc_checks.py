"""The checks of the arcs that the device makes as it narrows their ids, at the
edges of its 4,096-arc pieces: what they find is refused with the host check's
message, and what the host check accepts is accepted."""
import numpy as np
import pytest

from parity import assert_runs_equal, run_gpu, run_oracle

pytestmark = pytest.mark.gpu

N, D = 1500, 6          # a ring lattice: 9,000 arcs, three pieces


def _lattice():
    col = (np.arange(N)[:, None] + np.array([-3, -2, -1, 1, 2, 3])) % N
    col.sort(axis=1)
    return np.arange(N + 1, dtype=np.int64) * D, col.reshape(-1).astype(np.int64), np.ones(N * D)


@pytest.mark.parametrize("at", [0, 4095, 4096, N * D - 1])
@pytest.mark.parametrize("what", ["high", "low", "nan", "inf", "large"])
def test_a_bad_arc_is_named(at, what):
    import nido_amd as na
    off, col, w = _lattice()
    if what in ("high", "low"):
        col[at] = N if what == "high" else -1
        msg = rf"col\[{at}\]={col[at]} out of range"
    else:
        w[at] = {"nan": np.nan, "inf": -np.inf, "large": 2.0 ** 62}[what]
        msg = rf"weight\[{at}\] is not finite"
    print(f"case: {what} at {at}", flush=True)
    with pytest.raises(na.NidoError, match=msg):
        na.GraphGPU((off, col, w), 2)


@pytest.mark.parametrize("graph,at", [(0, 0), (1, 4095), (2, N * D - 1)])
def test_an_arc_that_leaves_its_graph_is_named(graph, at):
    import nido_amd as na
    off, col, w = _lattice()
    vptr, boff, bcol, bw = na.concat_graphs([(off, col, w)] * 3)
    e = graph * N * D + at
    bcol[e] = (graph + 1) % 3 * N + 5
    print(f"case: arc {e} of graph {graph}", flush=True)
    with pytest.raises(na.NidoError, match=rf"arc {e} \(col {bcol[e]}\) leaves graph {graph}"):
        na.BatchGPU(csr=(vptr, boff, bcol, bw), nbatches=2)


@pytest.mark.parametrize("scale,ok", [(2.0 ** 48, True), (2.0 ** 49, False)])
def test_the_total_is_decided_exactly(scale, ok):
    """9,000 weights: of 2^48 a total of 2^61.1, of 2^49 one of 2^62.1."""
    import nido_amd as na
    off, col, w = _lattice()
    w *= scale
    print(f"case: weights of {scale}", flush=True)
    if not ok:
        with pytest.raises(na.NidoError, match="total of"):
            na.GraphGPU((off, col, w), 2)
        return
    na.GraphGPU((off, col, w), 2).close()


def test_negative_weights_and_negative_zero():
    off, col, w = _lattice()
    src = np.repeat(np.arange(N), D)
    w[(src + col) % 7 == 0] = -0.25
    w[(src + col) % 11 == 0] = -0.0
    assert_runs_equal(run_oracle(off, col, w, 4), run_gpu(off, col, w, 4))
