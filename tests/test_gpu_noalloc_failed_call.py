"""A call of nido_modularity_noalloc that fails half-way leaves nothing behind
for the next one: bad input is flagged, the launch that would have reported it
fails, and the next call on good input gives that input's modularity."""
import pytest

from shim import run_with_shim

pytestmark = pytest.mark.gpu

CODE = """
import numpy as np
from test_zz_no_alloc import _hip, _reference
off, col, w = na.gen_sbm(1000, 50, 0.3, 0.01, True, 3).arrays()
q0, q1, comm = _reference(na, off, col, w, 2)
hip = _hip()
bad_col, bad_comm = col.copy(), comm.copy()
bad_col[-1] = len(off) - 1
bad_comm[7] = -1
dev, got = [], np.zeros(1)
for x in (off, col, w, comm, bad_col, bad_comm, got):
    p = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(p), x.nbytes) == 0
    dev.append(p.value)
    assert hip.hipMemcpy(p.value, x.ctypes.data, x.nbytes, 1) == 0
assert hip.hipDeviceSynchronize() == 0
d_off, d_col, d_w, d_comm, d_bad_col, d_bad_comm, d_q = dev

def q(cols, c):
    na.modularity_noalloc(len(off) - 1, len(col), d_off, cols, d_w, c, d_q, 0)
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemcpy(got.ctypes.data, d_q, 8, 2) == 0
    return float(got[0])

assert q(d_col, d_comm) == q1
for cols, c in ((d_bad_col, d_comm), (d_col, d_bad_comm)):
    # the k-th launch of the call fails, and those after it up to n in all (more
    # than the call has: the clean-up's too)
    for k, n in ((1, 1), (2, 1), (3, 1), (4, 1), (2, 4), (4, 2)):
        shim.shim_fail_launch(k, n)
        try:
            q(cols, c)
        except na.NidoError:
            pass
        else:
            raise SystemExit("the failed launch was not reported")
        shim.shim_fail_launch(0, 0)
        assert hip.hipDeviceSynchronize() == 0
        assert q(d_col, d_comm) == q1, (k, n, float(got[0]), q1)
    assert np.isnan(q(cols, c))
print("ok")
"""


def test_a_failed_call_leaves_no_flag(tmp_path):
    print("case: bad input, then a failed launch, then good input", flush=True)
    assert "ok" in run_with_shim(CODE, tmp_path)
