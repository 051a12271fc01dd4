"""qol_getnearquad_lap_rrq_mex_ keeps one whole-surface engine between calls: a
call gives the same triplets bit for bit whatever ran before it (another
geometry of the same shape, another shape or order, a refused call, fewer pairs)
and whatever runs beside it on other threads."""
import threading

import numpy as np
import pytest

from qotential_amd import rrq as R
from qotential_amd import workload as W

pytestmark = pytest.mark.gpu


def _job(p, scale, near, mp=4, np_=8):
    geo = W.geometry(mp, np_, p, modes=W.VMEC_BENCH)
    for k in ("sx", "rts", "rps"):
        geo[k] = geo[k] * scale
    geo["sw"] = geo["sw"] * scale ** 2
    n = geo["ntri"]
    rng = np.random.default_rng(p + near)
    rows = np.arange(n)[:, None] * geo["h"] + rng.integers(0, geo["h"], (n, near))
    tcx = geo["sx"][rows.ravel()] + 1e-3 * scale * geo["snx"][rows.ravel()]
    return geo, tcx, rows.ravel() + 1, 1 + near * np.arange(n + 1)


def test_calls_do_not_see_each_other():
    jobs = [_job(4, 1.0, 5), _job(4, 1.7, 5), _job(4, 1.0, 2), _job(6, 1.0, 5), _job(4, 1.0, 5, 6, 8)]
    first = [R.getnearquad_lap_rrq(*j) for j in jobs]

    def same(i):
        return all(np.array_equal(a, b) for a, b in zip(R.getnearquad_lap_rrq(*jobs[i]), first[i]))

    for i in (0, 1, 0, 2, 0, 3, 0, 4, 4, 0):
        assert same(i), i
    geo, tcx, row, tcxi = jobs[0]
    bad = tcxi.copy()
    bad[3] = bad[5] + 1
    with pytest.raises(Exception):
        R.getnearquad_lap_rrq(geo, tcx, row, bad)
    assert same(0)
    out = {}
    ts = [threading.Thread(target=lambda i=i: out.__setitem__(i, [same(i % 3) for _ in range(4)])) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert all(all(v) for v in out.values()) and len(out) == 4
