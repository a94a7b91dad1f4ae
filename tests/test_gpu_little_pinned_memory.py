"""Where only a page of pinned memory is to be had, handles copy through
pageable memory and give the same results: one graph with its lists built on
the host and on the device, and many graphs in one handle."""
import pytest

from shim import run_with_shim

pytestmark = pytest.mark.gpu

CODE = """
import numpy as np
from parity import assert_runs_equal, run_gpu, run_oracle
shim.shim_pinned_max.argtypes = [ctypes.c_size_t]
shim.shim_pinned_max(4096)
graph = na.gen_rmat(14, 16, 0.57, 0.19, 0.19, True, 7).arrays()
expected = run_oracle(*graph, 4)
for lists in (0, 1):
    na.set_device_lists(lists)
    assert_runs_equal(expected, run_gpu(*graph, 4))
na.set_device_lists(0)
graphs = [na.gen_sbm(n, 50, 0.3, 0.01, True, n).arrays() for n in (100, 2000, 1)]
b = na.BatchGPU(graphs, 2)
b.run()
for i, g in enumerate(graphs):
    assert np.array_equal(b.clustering(i), run_oracle(*g, 2)["clustering"])
b.close()
try:
    na.GraphGPU(graph, 4, window=len(graph[1]) // 2)   # its arcs stay in pinned memory
except na.NidoError as e:
    print("refused:", e)
else:
    raise SystemExit("no error")
print("ok")
"""


def test_handles_without_a_pinned_block(tmp_path):
    print("case: 4,096 bytes of pinned memory at a time", flush=True)
    assert run_with_shim(CODE, tmp_path).endswith("ok\n")
