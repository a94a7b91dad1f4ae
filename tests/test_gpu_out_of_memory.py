"""A handle whose allocations fail takes what other handles have freed, also
those that are still there: with room for little more than a first handle
holds, a second one is made and run, and both give what they give alone."""
import pytest

from shim import run_with_shim

pytestmark = pytest.mark.gpu

CODE = """
import numpy as np
shim.shim_pool_used.restype = ctypes.c_size_t
shim.shim_pool_limit.argtypes = [ctypes.c_size_t]

def lattice(n):
    k = np.concatenate([np.arange(-10, 0), np.arange(1, 11)])
    return np.arange(n + 1, dtype=np.int64) * 20, ((np.arange(n)[:, None] + k) % n).reshape(-1), np.ones(20 * n)

def run(g):
    st = na.LouvainGPU(500, 1e-6, 8).run(g)
    return st.q, g.clustering()

small = lattice(50_000)
with_room = na.GraphGPU(small, 8)
expected = run(with_room)
with_room.close()
a = na.GraphGPU(lattice(400_000), 8)      # its first coarse graph frees 130 MB
first = run(a)
held = shim.shim_pool_used()
shim.shim_pool_limit(held + (1 << 20))
graphs = [na.GraphGPU(small, 8) for _ in range(2)]
for b in graphs:
    got = run(b)
    assert got[0] == expected[0] and np.array_equal(got[1], expected[1])
assert shim.shim_pool_used() <= held + (1 << 20)
try:
    na.GraphGPU(lattice(2_000_000), 8)    # more than there is in any case
except na.NidoError as e:
    print("refused:", e)
else:
    raise SystemExit("no error")
b = na.GraphGPU(small, 8)
got = run(b)
assert got[0] == expected[0] and np.array_equal(got[1], expected[1])
assert np.array_equal(a.clustering(), first[1])
shim.shim_pool_limit(0)
for g in [a, b] + graphs:
    g.close()
print("ok")
"""


def test_a_second_handle_takes_what_the_first_one_freed(tmp_path):
    print("case: 1 MiB more than a handle of 8 M arcs holds", flush=True)
    assert run_with_shim(CODE, tmp_path).endswith("ok\n")
