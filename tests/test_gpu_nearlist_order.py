"""The brute-force near list with panels in random order, whose groups of 16 hold
most targets: the same pairs as with the panels in order, panel by panel; panel
counts that leave the last set of 64 part empty, short and several segments."""
import numpy as np
import pytest

from qotential_amd import workload as W
from qotential_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _pairs(geo, tx, radius):
    e = Engine(geo)
    e.set_targets(tx)
    e.set_near_radius(radius)
    e.nearlist()
    offs, idx = e.pairs()
    e.close()
    return [idx[a:b] for a, b in zip(offs[:-1], offs[1:])]


@pytest.mark.parametrize("npan,nt,radius", [(385, 9001, 0.0), (385, 63, 2.0), (193, 4097, 0.0), (15, 700, 2.0)])
def test_random_order(npan, nt, radius):
    geo = W.geometry(8, 20, 3, modes=W.VMEC_BENCH)
    h = geo["h"]
    tx = W.targets(geo, nt, -4.0, 0.5, sides=0, seed=npan)[0]
    tx[nt // 3] = np.nan
    perm = np.random.default_rng(nt).permutation(geo["ntri"])[:npan]

    def part(order):
        rows = (order[:, None] * h + np.arange(h)).ravel()
        return dict({k: np.ascontiguousarray(geo[k][rows]) for k in ("sx", "snx", "sw", "rts", "rps")}, p=3)

    mixed, ordered = _pairs(part(perm), tx, radius), _pairs(part(np.sort(perm)), tx, radius)
    rank = np.argsort(np.argsort(perm))
    assert sum(map(len, mixed)) > nt // 4
    assert all(np.array_equal(mixed[i], ordered[rank[i]]) for i in range(npan))
