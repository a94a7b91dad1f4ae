"""Hubs most of whose arcs lead into a few communities: the key fill of rows of
16 partitions (14,017 arcs) and more sums such arcs per wavefront.  Whole runs
against the oracle, with weights whose sums need one and two FP64 entries."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _hubs(leaves, groups, singles, weights, seed):
    """Two hubs joined to every leaf; leaves in `groups` stars of their own and
    `singles` more leaves without one."""
    rng = np.random.default_rng(seed)
    n = leaves + singles
    nv = 2 + groups + n
    first = 2 + groups
    leaf = first + np.arange(n)
    centre = 2 + rng.integers(groups, size=leaves)
    u = np.concatenate([np.zeros(n, np.int64), np.ones(n, np.int64), centre, [0]])
    v = np.concatenate([leaf, leaf, leaf[:leaves], [1]])
    m = len(u)
    if weights == "unit":
        w = np.ones(m)
    else:
        w = rng.integers(1, 1 << 51, m) / float(1 << 53)            # up to 1/4, multiples of 2^-53
        w[2 * n:] = 1.0                                             # the stars hold together
        if weights == "signed":
            w[:2 * n:7] *= -1.0
    r, c, ww = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    order = np.lexsort((c, r))
    off = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=nv))]).astype(np.int64)
    return off, c[order].astype(np.int64), ww[order]


@pytest.mark.parametrize("leaves,groups,singles", [
    (13138, 1, 0),               # just below and above 16 partitions
    (14017, 3, 0),
    (30000, 12, 40),             # as many heavy communities as are looked for
    (18000, 200, 2000),          # none that many of 64 arcs share
])
@pytest.mark.parametrize("weights", ["unit", "fractions", "signed"])
def test_hubs_into_few_communities(leaves, groups, singles, weights):
    from parity import assert_runs_equal, run_gpu, run_oracle
    off, col, w = _hubs(leaves, groups, singles, weights, leaves + groups)
    print(f"case: {leaves} leaves, {groups} groups, {singles} singles, {weights}", flush=True)
    assert_runs_equal(run_oracle(off, col, w, 4), run_gpu(off, col, w, 4))
