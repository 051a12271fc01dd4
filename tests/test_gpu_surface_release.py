"""The whole-surface engine that qol_getnearquad_lap_rrq_mex_ keeps: its device
memory is given back by qol_clear_patch_levels_all_mex_, and by the next call of
another shape before that call makes its own engine (a call refused afterwards
therefore leaves nothing behind)."""
import ctypes as C

import numpy as np
import pytest

from qotential_amd import rrq as R
from qotential_amd import workload as W
from qotential_amd._lib import QolError, lib

pytestmark = pytest.mark.gpu
MB = 1 << 20


def _free():
    a, b = C.c_size_t(), C.c_size_t()
    assert lib().hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


def _job(p, near):
    geo = W.geometry(8, 20, p, modes=W.VMEC_BENCH)
    n, h = geo["ntri"], geo["h"]
    rows = (np.arange(n)[:, None] * h + np.arange(near) % h).ravel()
    return geo, geo["sx"][rows] + 1e-3 * geo["snx"][rows], rows + 1, 1 + near * np.arange(n + 1)


def test_kept_engine_is_given_back():
    big, small = _job(6, 300), _job(4, 2)
    R.getnearquad_lap_rrq(*small)  # whatever a first call sets up for good
    R.clear_patch_levels_all()
    free = _free()
    want = R.getnearquad_lap_rrq(*big)
    # per pair, 4 columns of triplets and 5 moment vectors of 21, 2 of them weights: 1.8 KB
    assert free - _free() > 150 * MB
    assert R.clear_patch_levels_all() == 0
    assert abs(free - _free()) < 16 * MB
    assert all(np.array_equal(a, b) for a, b in zip(R.getnearquad_lap_rrq(*big), want))
    geo, tcx, row, tcxi = small
    bad = tcxi.copy()
    bad[3] = bad[5] + 1
    with pytest.raises(QolError):
        R.getnearquad_lap_rrq(geo, tcx, row, bad)
    assert abs(free - _free()) < 16 * MB
    assert all(np.array_equal(a, b) for a, b in zip(R.getnearquad_lap_rrq(*big), want))
    R.clear_patch_levels_all()
