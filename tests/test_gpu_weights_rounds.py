"""RRQ weights at the edges of the weights kernels' rounds of 32 pairs, on both
sides of the order above which the operator is formed first: calls on the first
31, 32, 33 and 65 targets of a panel against one call on all, bit for bit, and
their action on a smooth density against the oracle.  The bounds on the action
interpolate (geometrically) between those of orders 8 and 12, 1e-10 and 4e-7,
that the rounding of the panel systems, conditioned 2e10 at order 12, sets."""
import numpy as np
import pytest

from qotential_amd import workload as W
from qotential_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,tol", [(3, 1e-10), (8, 1e-10), (9, 8e-10), (10, 7e-9), (11, 5e-8), (12, 4e-7)])
def test_rounds_and_operator(p, tol, oracle):
    geo = W.geometry(8, 20, p, modes=W.VMEC_BENCH)
    h = geo["h"]
    ub, gu = W.charge_field(geo["sx"], *W.point_charges(geo, seed=3))
    sl = slice(7 * h, 8 * h)
    ub, ubn = ub[sl], (geo["snx"] * gu).sum(1)[sl]
    one = {k: np.ascontiguousarray(geo[k][sl]) for k in ("sx", "snx", "sw", "rts", "rps")}
    one.update(p=p, ntri=1)
    tx = W.targets(one, 150, -3.0, -1.0, sides=0, seed=p)[0]
    e = Engine(one)
    e.force_label(5)

    def weights(n):
        e.set_targets(tx[:n])
        e.set_pairs(np.array([0, n]), 1 + np.arange(n))
        e.eval()
        return e.weights()

    full = weights(150)
    for n in (31, 32, 33, 65):
        w = weights(n)
        for k in ("As", "Ad"):
            assert np.array_equal(w[k], full[k][:n]), (n, k)
    e.close()
    oracle.set_side_tol(1e-10)
    try:
        o = oracle.rrq(p, tx, one["sx"], one["snx"], one["sw"], one["rts"], one["rps"], exterior=True)
    finally:
        oracle.set_side_tol(1e300)
    rr = o["label"] == 5
    assert rr.sum() > 10
    act = np.abs((full["As"] - o["As"]) @ ubn - (full["Ad"] - o["Ad"]) @ ub)
    act /= np.abs(o["As"]) @ np.abs(ubn) + np.abs(o["Ad"]) @ np.abs(ub)
    assert act[rr].max() < tol, act[rr].max()
