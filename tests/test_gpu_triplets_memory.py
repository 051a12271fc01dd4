"""An engine's triplets leave no device memory behind: their columns (32 h bytes a
pair) are the call's own, and a later call gives the same triplets."""
import ctypes as C

import numpy as np
import pytest

from qotential_amd import workload as W
from qotential_amd._lib import lib
from qotential_amd.engine import Engine

pytestmark = pytest.mark.gpu
MB = 1 << 20


def _free():
    a, b = C.c_size_t(), C.c_size_t()
    assert lib().hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


def test_triplets_give_their_buffers_back():
    p, nt = 6, 20000
    geo = W.geometry(8, 20, p, modes=W.VMEC_BENCH)
    e = Engine(geo)
    e.set_targets(W.targets(geo, nt, -4.0, -1.0, sides=0, seed=1)[0])
    e.nearlist()
    e.eval()
    e.sync()
    free = _free()
    first = e.triplets(1 + np.arange(nt))
    assert 32 * e.h * e.nnz > 64 * MB
    assert free - _free() < 16 * MB
    assert all(np.array_equal(a, b) for a, b in zip(e.triplets(1 + np.arange(nt)), first))
    e.close()
