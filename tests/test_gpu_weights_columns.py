"""Fetching the weights of a levels-only evaluation: the columns pass through a
device buffer of bounded size, so many columns at a time (the moment vectors'
buffer, which holds them all after a whole evaluation, does not exist then).  The
weights are those of a whole evaluation of the same pairs, bit for bit; the device
memory a large call leaves behind is its weights and little more."""
import ctypes as C
import threading

import numpy as np
import pytest

from qotential_amd import rrq as R
from qotential_amd import workload as W
from qotential_amd._lib import lib
from qotential_amd.engine import Engine

pytestmark = pytest.mark.gpu
MB = 1 << 20


def _free():
    a, b = C.c_size_t(), C.c_size_t()
    assert lib().hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


# weights of 2h doubles a target: 16 MB hold all columns, all but one, 29 of 72 (so that
# a pass takes columns of both matrices), 5 of 12 and 20 of 72
@pytest.mark.parametrize("p,m", [(8, 29000), (8, 29200), (8, 70001), (3, 400000), (8, 100000)])
def test_columns_and_memory(p, m):
    geo = W.geometry(8, 20, p, modes=W.VMEC_BENCH)
    h = geo["h"]
    one = {k: np.ascontiguousarray(geo[k][5 * h:6 * h]) for k in ("sx", "snx", "sw", "rts", "rps")}
    one.update(p=p, ntri=1)
    tx = W.targets(one, m, -0.5, 1.0, sides=0, seed=m)[0]
    e = Engine(one)
    e.set_targets(tx)
    e.set_pairs(np.array([0, m]), 1 + np.arange(m))
    e.eval()
    w = e.weights()
    e.close()
    lv, ier = R.build_patch_levels(one["sx"], one["rts"], one["rps"], p - 1)
    assert ier == 0
    out = {}

    def call():  # on a thread of its own: the engine kept per thread is a new one
        free = _free()
        out["r"] = R.lap3dsdlpmat_levels(tx, h, lv)
        out["held"] = free - _free()

    try:
        t = threading.Thread(target=call)
        t.start()
        t.join()
    finally:
        R.clear_patch_levels(lv)
    As, Ad, idxs, ier = out["r"]
    served = w["label"] <= 4
    assert ier == 0 and np.array_equal(idxs, 1 + np.nonzero(~served)[0]) and served.sum() > m // 10
    assert np.array_equal(As[served], w["As"][served]) and np.array_equal(Ad[served], w["Ad"][served])
    # weights, the targets and lists (60 bytes a target), the panel and its order's tables (below 16 MB)
    assert out["held"] < 16 * h * m + 100 * m + (16 + 16) * MB
