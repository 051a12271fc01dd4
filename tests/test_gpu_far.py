"""Far-field direct sum (far.hip) against numpy at the edges of its plan: one,
two and four targets per thread, partial tiles, one and several source chunks,
coincident points, and coordinates the sum has to leave out."""
import numpy as np
import pytest

from qotential_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _cloud(npan, seed):
    rng = np.random.default_rng(seed)
    n = 3 * npan  # order 2: three nodes a panel
    nx = rng.standard_normal((n, 3))
    nx /= np.linalg.norm(nx, axis=1)[:, None]
    geo = dict(p=2, sx=rng.uniform(-1, 1, (n, 3)), snx=nx, sw=rng.uniform(0.1, 1, n), rts=rng.standard_normal((n, 3)),
               rps=rng.standard_normal((n, 3)))
    return geo, rng.standard_normal(n), rng.standard_normal(n), rng


def _sum(geo, tx, ub, ubn):
    """the sum and, for the tolerance, the sum of the terms' magnitudes"""
    d = tx[:, None, :] - geo["sx"][None]
    rr = (d * d).sum(-1)
    on = rr > 1e-28
    ri = np.where(on, 1.0 / np.sqrt(np.where(on, rr, 1.0)), 0.0)
    w = geo["sw"] / (4 * np.pi)
    v = w * (ubn * ri - ub * (d * geo["snx"][None]).sum(-1) * ri ** 3)
    return v.sum(1), (w * (np.abs(ubn) * ri + np.abs(ub) * ri ** 2)).sum(1)


@pytest.mark.parametrize("nt,npan", [(1, 1), (64, 11), (65, 500), (256, 11), (257, 2000), (4099, 371)])
def test_far_vs_numpy(nt, npan):
    print("far", nt, npan, flush=True)
    geo, ub, ubn, rng = _cloud(npan, nt)
    tx = rng.uniform(-1.2, 1.2, (nt, 3))
    tx[:: 7] = geo["sx"][rng.integers(0, 3 * npan, len(tx[:: 7]))]  # coincident with a source
    e = Engine(geo)
    e.set_targets(tx)
    u = e.far(ub, ubn)
    ref, mag = _sum(geo, tx, ub, ubn)
    # every term to 16 roundings, every sum at most 3 npan additions deep (both sides)
    assert np.all(np.abs(u - ref) <= (6 * npan + 16) * 2.3e-16 * mag)
    assert np.array_equal(u, e.far(ub, ubn))


def test_far_left_out():
    """a NaN position contributes nothing, a huge one nothing, an infinite target gives NaN"""
    geo, ub, ubn, rng = _cloud(40, 5)
    tx = rng.uniform(-1.2, 1.2, (70, 3))
    ref, mag = _sum(dict(geo, sw=np.where(np.arange(120) % 60 == 8, 0.0, geo["sw"])), tx, ub, ubn)
    geo["sx"][8, 1] = np.nan
    geo["sx"][68, 2] = 1e170
    e = Engine(geo)
    tx[3, 0], tx[5, 1], tx[66, 2] = np.nan, np.inf, -1e160
    e.set_targets(tx)
    u = e.far(ub, ubn)
    assert u[3] == 0.0 and u[66] == 0.0 and np.isnan(u[5])
    ok = np.ones(70, bool)
    ok[[3, 5, 66]] = False
    assert np.all(np.abs(u - ref)[ok] <= 256 * 2.3e-16 * mag[ok])


def _plain(geo, tx, ub, ubn):
    """the formula term by term: whatever a term is, infinite or not a number, it counts
    unless its r^2 is not above the threshold"""
    with np.errstate(all="ignore"):
        d = tx[:, None, :] - geo["sx"][None]
        rr = (d * d).sum(-1)
        ri = 1.0 / np.sqrt(rr)
        w = geo["sw"] / (4 * np.pi)
        v = w * ubn * ri - w * ub * (d * geo["snx"][None]).sum(-1) * ri * ri * ri
        return np.where(rr > 1e-28, v, 0.0).sum(1)


@pytest.mark.parametrize("nt,npan", [(5, 1), (40, 11), (200, 11), (300, 700)])
def test_far_out_of_range(nt, npan):
    """far coordinates whose squares still fit count in full, and a node's own strength
    never reaches the target on it, whatever else is infinite or not a number: targets by
    one, two and four a thread, one and several chunks"""
    geo, ub, ubn, rng = _cloud(npan, 9 * nt)
    ns = 3 * npan
    tx = rng.uniform(-1.2, 1.2, (nt, 3))

    def check(geo, tx, ub, ubn):
        e = Engine(geo)
        e.set_targets(tx)
        u = e.far(ub, ubn)
        e.close()
        ref = _plain(geo, tx, ub, ubn)
        fin = np.isfinite(ref)
        assert np.array_equal(u[~fin], ref[~fin], equal_nan=True)
        # each side: 16 roundings a term, ns additions (see test_far_vs_numpy), no
        # cancellation: the strengths of one sign, or one term alone
        assert np.all(np.abs(u[fin] - ref[fin]) <= (2 * ns + 16) * 2.3e-16 * np.abs(ref[fin]))

    zero, one = np.zeros(ns), rng.uniform(0.5, 1.0, ns)
    far_t = tx.copy()
    far_t[::2, 1] = 10.0 ** rng.uniform(149.5, 153.5, len(far_t[::2]))
    check(geo, far_t, zero, one)
    far_s = dict(geo, sx=geo["sx"].copy())
    far_s["sx"][ns - 1] = 1e152, 2e152, -3e151
    check(far_s, tx, zero, np.where(np.arange(ns) == ns - 1, 1.0, 0.0))
    check(far_s, tx, zero, one)
    for bad in (np.nan, np.inf, -np.inf):
        on = tx.copy()
        on[::3] = geo["sx"][1]
        b = one.copy()
        b[1] = bad
        check(geo, on, zero, b)
        nx = np.tile([0.0, 0.0, 1.0], (ns, 1))  # an infinite strength times the normal's zeros
        flat = dict(geo, snx=nx, sx=geo["sx"] * [1, 1, 0] - [0, 0, 2.0])
        d = one.copy()
        d[1] = bad
        check(flat, tx, d, zero)
    lost = dict(geo, sx=geo["sx"].copy())
    lost["sx"][2, 0] = np.nan
    b = one.copy()
    b[2] = np.nan
    check(lost, tx, zero, b)
    check(geo, tx, zero, 1e308 * one)
