"""Near corrections of orders 2 to 6, on both sides of the node count up to which
four lanes take a pair, against numpy: groups of 64 pairs (32 above) filled by one
panel, by more panels than a workgroup gathers, and left over; the values fused
into eval against those of apply.  The bound is that of test_gpu_apply_groups."""
import numpy as np
import pytest

from qotential_amd import workload as W
from qotential_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("per_panel", [[1], [63], [64, 1], [65, 0, 3], [1] * 130, [0, 5, 40] * 5])
def test_small_orders_vs_numpy(p, per_panel):
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
    u, val = e.apply(ub, ubn, np.zeros(len(k)))
    e.eval()  # the density is resident now: eval forms the values itself
    fused = e.values()[0]
    e.close()
    node = k[:, None] * h + np.arange(h)
    d = tx[:, None] - geo["sx"][node]
    r = np.sqrt((d * d).sum(2))
    s = geo["sw"][node] / (4 * np.pi * r)
    dl = s * (d * geo["snx"][node]).sum(2) / r ** 2
    terms = np.concatenate([(w["As"] - s) * ubn[node], -(w["Ad"] - dl) * ub[node]], axis=1)
    mag = ((np.abs(w["As"]) + s) * np.abs(ubn[node]) + (np.abs(w["Ad"]) + s / r) * np.abs(ub[node])).sum(1)
    assert (np.abs(val - terms.sum(1)) <= 1e-13 * mag).all()
    assert np.array_equal(fused, val) and np.array_equal(u, val)
