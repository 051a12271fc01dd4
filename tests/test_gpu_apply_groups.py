"""Near corrections against numpy at the edges of the apply kernels' groups of 32
pairs: one pair, 31 to 33, groups whose pairs belong to more panels than a
workgroup gathers, panels without pairs, and orders whose node counts leave
lanes over.  The bound is 1e-13 of the sum of the terms' magnitudes (at most 156
terms; the naive entries' reciprocal root is good to 2 ulp, and the product of
distance and normal is taken at its factors' size)."""
import numpy as np
import pytest

from qotential_amd import workload as W
from qotential_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,per_panel", [(3, [1]), (4, [31]), (4, [32]), (6, [33, 0, 1]), (8, [1] * 70), (8, [0, 5, 40] * 4),
                                         (12, [3] * 30), (12, [64, 1])])
def test_groups_vs_numpy(p, per_panel):
    geo = W.geometry(8, 20, p, modes=W.VMEC_BENCH)
    h, rng = geo["h"], np.random.default_rng(p + len(per_panel))
    counts = np.zeros(geo["ntri"], dtype=int)
    counts[:len(per_panel)] = per_panel
    k = np.repeat(np.arange(geo["ntri"]), counts)
    g = k * h + rng.integers(0, h, len(k))
    tx = geo["sx"][g] + geo["snx"][g] * 10 ** rng.uniform(-2, 0.5, (len(k), 1)) * np.sqrt(geo["sw"][:h].sum())
    ub, ubn = rng.standard_normal((2, geo["ntri"] * h))
    e = Engine(geo)
    e.set_targets(tx)
    e.set_pairs(np.concatenate([[0], np.cumsum(counts)]), 1 + np.arange(len(k)))
    e.eval()
    w = e.weights()
    u0 = rng.standard_normal(len(k))
    u = e.apply(ub, ubn, u0)[0]
    e.close()
    node = k[:, None] * h + np.arange(h)
    d = tx[:, None] - geo["sx"][node]
    r = np.sqrt((d * d).sum(2))
    s = geo["sw"][node] / (4 * np.pi * r)
    dl = s * (d * geo["snx"][node]).sum(2) / r ** 2
    terms = np.concatenate([(w["As"] - s) * ubn[node], -(w["Ad"] - dl) * ub[node]], axis=1)
    mag = (np.abs(w["As"]) + s) * np.abs(ubn[node]) + (np.abs(w["Ad"]) + s / r) * np.abs(ub[node])
    err = np.abs(u - u0 - terms.sum(1))
    assert (err <= 1e-13 * mag.sum(1) + 1e-15 * np.abs(u0)).all(), (err / mag.sum(1)).max()
