"""The brute-force near list against numpy's own loop over panels (the same
sums, so the same list): panel counts around the waves' 64 and the groups' 16,
target counts around the wave and the segments, a far group, a panel that every
target is near, a ball and targets that are not numbers or infinite."""
import numpy as np
import pytest

from qotential_amd import workload as W
from qotential_amd.engine import Engine

pytestmark = pytest.mark.gpu


def ball_rule(sx, sw, npan, tx):
    h = len(sw) // npan
    offs, idx = [0], []
    for k in range(npan):
        q, s = np.zeros(3), 0.0
        for i in range(h):
            q = q + sx[k * h + i]
            s = s + sw[k * h + i]
        q, r = q / h, 1.75 * np.sqrt(s)
        d = tx - q
        idx.append(1 + np.nonzero(d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2] < r * r)[0])
        offs.append(offs[-1] + len(idx[-1]))
    return np.array(offs), np.concatenate(idx)


@pytest.mark.parametrize("npan,nt", [(1, 1), (1, 64), (15, 65), (16, 4097), (17, 63), (63, 4096), (64, 129), (65, 5000),
                                     (320, 9001)])
def test_groups_vs_numpy(npan, nt):
    p, rng = 3, np.random.default_rng(npan + nt)
    geo = W.geometry(8, 20, p, modes=W.VMEC_BENCH)
    h = geo["h"]
    part = {k: np.ascontiguousarray(geo[k][:npan * h]) for k in ("sx", "snx", "sw")}
    part.update({k: geo[k][:npan * h] for k in ("rts", "rps")}, p=p, ntri=npan)
    sw = part["sw"] = part["sw"].copy()
    if npan > 16:
        sw[16 * h:17 * h] = 1e3       # near to every target
    if npan > 20:
        sw[19 * h] = np.nan           # near to none
        sw[20 * h:21 * h] = np.inf    # to every finite one
    tx = geo["sx"][rng.integers(0, npan * h, nt)] + rng.normal(0.0, 0.1, (nt, 3)) * rng.random((nt, 1)) ** 4
    tx[rng.random(nt) < 0.2] += 5.0
    if nt > 100:
        tx[[3, 70], [0, 2]] = np.nan
        tx[[5, 99], 1] = np.inf
    e = Engine(part)
    e.set_targets(tx)
    e.nearlist()
    offs, idx = e.pairs()
    e.close()
    with np.errstate(invalid="ignore"):
        ro, ri = ball_rule(part["sx"], sw, npan, tx)
    assert np.array_equal(offs, ro) and np.array_equal(idx, ri)
