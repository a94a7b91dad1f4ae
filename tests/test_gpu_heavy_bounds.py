"""The key fill's sums of heavy communities at their bounds: rows of 15, 16 and 17
partitions (13,140 / 13,141 and 14,016 / 14,017 arcs), and weights that a short
row sums in fixed point but a wavefront of the key fill does not.  Whole runs
against the oracle."""
import numpy as np
import pytest

from parity import assert_runs_equal, run_gpu, run_oracle
from test_gpu_heavy_communities import _hubs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("arcs", [13140, 13141, 14016, 14017])
@pytest.mark.parametrize("weights", ["unit", "signed"])
def test_rows_around_sixteen_partitions(arcs, weights):
    off, col, w = _hubs(arcs - 1, 3, 0, weights, arcs)      # a hub's arcs: the leaves and the other hub
    assert np.diff(off)[0] == arcs
    print(f"case: hubs of {arcs} arcs, {weights}", flush=True)
    assert_runs_equal(run_oracle(off, col, w, 4), run_gpu(off, col, w, 4))


@pytest.mark.parametrize("bits", [53, 54, 56])
@pytest.mark.parametrize("big_min_deg", [64, 512])
def test_weights_too_wide_for_a_wavefront_sum(bits, big_min_deg):
    """Weights up to 1 on a grid of 2^-bits: of 54 bits and more, 512 of them
    reach 2^63, 64 do not."""
    off, col, w = _hubs(20000, 3, 40, "unit", bits)
    lo = np.minimum(np.repeat(np.arange(len(off) - 1), np.diff(off)), col)
    hi = np.maximum(np.repeat(np.arange(len(off) - 1), np.diff(off)), col)
    w[(lo * 31 + hi) % 3 == 0] = 3.0 * 2.0 ** -bits
    w[(lo * 31 + hi) % 3 == 1] = 1.0 - 2.0 ** -40
    print(f"case: weights of {bits} bits, short rows up to {big_min_deg}", flush=True)
    assert_runs_equal(run_oracle(off, col, w, 4), run_gpu(off, col, w, 4, big_min_deg=big_min_deg))
