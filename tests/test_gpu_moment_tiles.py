"""RRQ weights of one panel's targets do not depend on how the moments kernel
deals the pairs to tiles and workgroups: one call on all targets (several tiles,
several workgroups) against calls on the first 1, 15, 16, 17 and 48 of them, bit
for bit, and against the oracle on the first ones."""
import numpy as np
import pytest

from qotential_amd import workload as W
from qotential_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,tol", [(2, 1e-11), (4, 1e-11), (7, 1e-8), (8, 2e-7), (9, 2e-7), (10, 2e-6), (12, None)])
def test_tiles_and_split(p, tol, oracle):
    geo = W.geometry(4, 8, p, modes=W.VMEC_BENCH)
    h = geo["h"]
    one = {k: np.ascontiguousarray(geo[k][5 * h:6 * h]) for k in ("sx", "snx", "sw", "rts", "rps")}
    one.update(p=p, ntri=1)
    tx = W.targets(one, 333, -5.0, -1.0, sides=0, seed=p)[0]
    e = Engine(one)
    e.force_label(5)

    def weights(n):
        e.set_targets(tx[:n])
        e.set_pairs(np.array([0, n]), 1 + np.arange(n))
        e.eval(want_omega=True)
        return e.weights(omega=True)

    full = weights(333)
    for n in (1, 15, 16, 17, 48):
        w = weights(n)
        for k in ("As", "Ad", "Ias"):
            assert np.array_equal(w[k], full[k][:n]), (n, k)
        assert np.array_equal(w["Omega"], full["Omega"][:, :n])
    if tol is None:
        return  # conditioning: the orders' own test bounds the action instead
    oracle.set_side_tol(1e-10)
    o = oracle.rrq(p, tx[:40], one["sx"], one["snx"], one["sw"], one["rts"], one["rps"], exterior=True)
    rr = o["label"] == 5
    assert rr.sum() > 3
    for k in ("As", "Ad"):
        err = np.abs(full[k][:40] - o[k])[rr] / np.abs(o[k][rr]).max(1)[:, None]
        assert err.max() < tol, (k, err.max())
    assert np.abs(full["Omega"][:, :40] - o["Omega"])[:, rr].max() < 1e-10 * np.abs(o["Omega"][:, rr]).max()
