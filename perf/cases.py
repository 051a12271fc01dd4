"""The work that a user of this framework has it do, as cases that can be timed.

Six kinds of call, each through a public entry point:

  rrq           rrq.rrq: the weights of one panel for its near targets, the call
                that the reference's drivers make once per panel.  Latency counts.
  getnearquad   rrq.getnearquad_lap_rrq: the COO triplets of a whole surface.
  layer         grf.layer_potential: the whole call on new targets (near list,
                far field, close evaluation, correction), the engine kept.
  step          one close evaluation and its scatter into the potential, with
                geometry, targets, near list, far field and density resident: the
                benchmark's step, by the ball rule ("plain"), with the learned
                selector, or with split precision.
  mixed         the same step for a surface with several patch orders
                (mixed.MixedBatch).
  closepanel    rrq.lap3ddlp_closepanel: the close double layer of a tensor patch.

Host arrays go in and out of the drop-in calls and of layer_potential, as their
callers have them.  The resident step returns the potential.
"""
import ctypes
import functools
import math

import numpy as np

from qotential_amd import grf, mixed, rrq
from qotential_amd import workload as W
from qotential_amd._lib import check, lib, ptr
from qotential_amd.engine import Engine, order_info
from qotential_amd.selector import MODEL_FILE, Selector

# Shares of the near pairs that the ball rule serves on levels 1 to 4 and by RRQ
# for targets at h 10^U, U in [-6, -1] (the 48 x 120, order-8 benchmark surface),
# and near pairs per target: what the counts of work() are estimated from.
SHARES = (0.40, 0.27, 0.11, 0.055, 0.165)
PAIRS_PER_TARGET = 9.8


def listed():
    return [
        # one panel's targets as the reference's bench driver calls it (order 4,
        # built-in surface, about 124 targets a panel): the smallest call
        dict(name="rrq_p4_m124", kind="rrq", mp=24, np=72, order=4, targets=124, exterior=True),
        # a busy panel at order 6, an odd number of targets
        dict(name="rrq_p6_m1501", kind="rrq", mp=16, np=40, order=6, targets=1501, exterior=False),
        # the MATLAB caller's sparse correction on a surface of the order-4 fixture's
        # size (159 pairs a panel there), lists from a nearest-neighbour search
        dict(name="getnearquad_p4", kind="getnearquad", mp=12, np=36, order=4, targets=8640, near=159, exterior=True),
        # the CPU reference configuration: order 4, 4,000 interior targets
        dict(name="layer_p4_4000", kind="layer", mp=16, np=40, order=4, targets=4000, sides=-1, chart=False),
        # an ordinary evaluation with the exact chart boundary, both sides, odd count
        dict(name="layer_p6_20011", kind="layer", mp=24, np=72, order=6, targets=20011, sides=0, chart=True),
        # new targets on the benchmark surface: the far field of 513,000 nodes included
        dict(name="layer_p8_50000", kind="layer", mp=48, np=120, order=8, targets=50000, sides=0, chart=False),
        # the benchmark step
        dict(name="step_p8_200000", kind="step", mp=48, np=120, order=8, targets=200000, sides=0, path="plain"),
        # its two other paths, on a smaller surface
        dict(name="step_p8_selector", kind="step", mp=24, np=60, order=8, targets=50003, sides=0, path="selector"),
        dict(name="step_p6_split", kind="step", mp=24, np=72, order=6, targets=60000, sides=0, path="split"),
        # the highest order
        dict(name="step_p12_30000", kind="step", mp=16, np=40, order=12, targets=30000, sides=0, path="plain"),
        # an order per chart, all orders launched from one call
        dict(name="mixed_4_to_12", kind="mixed", mp=32, np=80, orders="4,6,8,10,12", targets=60000),
        # the reference's tensor patch (order 8), targets from 1e-7 to 0.1 off it
        dict(name="closepanel_p8_777", kind="closepanel", order=8, targets=777, ref=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


SURFACES = ((12, 36), (16, 40), (24, 60), (24, 72), (32, 80), (48, 120))


def draw(rng):
    kind = rng.choice(("rrq", "rrq", "getnearquad", "layer", "layer", "layer", "step", "step", "step", "step", "mixed",
                       "closepanel"))
    if kind == "closepanel":
        return dict(kind=kind, order=rng.randint(4, 10), targets=_log_int(rng, 20, 2000), ref=rng.randint(0, 2))
    mp, np_ = rng.choice(SURFACES[:4] if kind in ("rrq", "getnearquad") else SURFACES)
    if kind == "rrq":
        return dict(kind=kind, mp=mp, np=np_, order=rng.randint(3, 6), targets=_log_int(rng, 16, 4000),
                    exterior=rng.random() < 0.5)
    if kind == "getnearquad":
        return dict(kind=kind, mp=mp, np=np_, order=rng.randint(3, 6), targets=_log_int(rng, 500, 8640),
                    near=_log_int(rng, 5, 200), exterior=rng.random() < 0.5)
    if kind == "mixed":
        orders = sorted(rng.sample((4, 5, 6, 7, 8, 9, 10, 12), rng.randint(2, 4)))
        return dict(kind=kind, mp=mp, np=np_, orders=",".join(map(str, orders)), targets=_log_int(rng, 1000, 60000))
    order = rng.randint(4, 8) if mp == 48 else rng.choice((3, 4, 5, 6, 7, 8, 9, 10, 11, 12))
    if kind == "layer":
        return dict(kind=kind, mp=mp, np=np_, order=order, targets=_log_int(rng, 100, 40000),
                    sides=rng.choice((-1, 0)), chart=rng.random() < 0.3)
    path = rng.choice(("plain", "plain", "plain", "selector", "split"))
    return dict(kind=kind, mp=mp, np=np_, order=order, targets=_log_int(rng, 500, 120000 if order <= 8 else 40000),
                sides=rng.choice((-1, 0)), path=path)


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=8)
def _surface(mp, np_, order):
    return W.geometry(mp, np_, order, modes=W.VMEC_BENCH)


@functools.lru_cache(maxsize=2)
def _mixed_surface(mp, np_, orders):
    return mixed.surface(mp, np_, orders, modes=W.VMEC_BENCH, seed=11)


def _charges(geo, seed):
    return W.point_charges(geo, nchg=8, offset=0.4, seed=seed)


def _field(geo, charges):
    ub, gu = W.charge_field(geo["sx"], *charges)
    return ub, (geo["snx"] * gu).sum(1)


def _panel_targets(geo, k, n, seed):
    """n targets above panel k and the twelve panels nearest to it"""
    h = geo["h"]
    c = geo["sx"].reshape(-1, h, 3).mean(1)
    near = np.argsort(((c - c[k]) ** 2).sum(1), kind="stable")[:13]
    rows = (near[:, None] * h + np.arange(h)).ravel()
    sub = dict(p=geo["p"], ntri=len(near), sx=np.ascontiguousarray(geo["sx"][rows]),
               snx=np.ascontiguousarray(geo["snx"][rows]))
    return W.targets(sub, n, -6.0, -1.0, sides=0, seed=seed)[0]


def _torus_patch(p):
    """the tensor patch of the reference's smoke test (test/test_lap3d_close.f90:44-73)"""
    t = np.polynomial.legendre.leggauss(p)[0]
    x1, x2 = np.meshgrid(0.5 * t, 0.25 * t)
    s = np.stack([0.5 * np.sin(x1), (1 + 0.5 * np.cos(x1)) * np.sin(x2), (1 + 0.5 * np.cos(x1)) * np.cos(x2)], -1)
    s = s.reshape(-1, 3)
    return s - s.mean(0)


def _targets(case, seed):
    geo = _surface(case["mp"], case["np"], case["order"])
    tx, _, dist = W.targets(geo, case["targets"], -6.0, -1.0, sides=case["sides"], seed=seed + 1)
    return geo, tx, dist


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind)
    if kind == "closepanel":
        p, rng = case["order"], np.random.default_rng(seed)
        sx, n = _torus_patch(p), case["targets"]
        off = 10.0 ** rng.uniform(-7, -1, n) * rng.choice([-1.0, 1.0], n)
        s.update(sx=sx, order=p, ref=case["ref"], tx=sx[rng.integers(0, p * p, n)] + off[:, None] * np.array([0.0, 0, 1]))
        return s
    if kind == "mixed":
        surf = _mixed_surface(case["mp"], case["np"], tuple(int(p) for p in case["orders"].split(",")))
        tx = mixed.targets(surf, case["targets"], -6.0, -1.0, sides=0, seed=seed + 1)[0]
        charges = _charges(next(iter(surf["parts"].values())), seed + 2)
        s["batch"] = mixed.MixedBatch(surf, tx, lambda x: W.charge_field(x, *charges))
        return s
    p = case["order"]
    if kind == "rrq":
        geo = _surface(case["mp"], case["np"], p)
        k, h = int(np.random.default_rng(seed).integers(geo["ntri"])), geo["h"]
        s.update(order=p, exterior=case["exterior"], pre=rrq.simplex_precomp(p + 2, p - 1),
                 tx=_panel_targets(geo, k, case["targets"], seed + 1))
        s.update({a: np.ascontiguousarray(geo[a][k * h:(k + 1) * h]) for a in ("sx", "snx", "sw", "rts", "rps")})
        return s
    if kind == "getnearquad":
        geo, tx, _ = _targets(dict(case, sides=0), seed)
        c = geo["sx"].reshape(geo["ntri"], -1, 3).mean(1)
        idx = np.concatenate([np.sort(np.argpartition(((tx - x) ** 2).sum(1), case["near"] - 1)[:case["near"]]) for x in c])
        s.update(geo=geo, tcx=np.ascontiguousarray(tx[idx]), tcxrow=idx + 1,
                 tcxi=1 + case["near"] * np.arange(geo["ntri"] + 1), iside=30 if case["exterior"] else 31)
        return s
    geo, tx, _ = _targets(case, seed)
    ub, ubn = _field(geo, _charges(geo, seed + 2))
    chart = W.chart_boundary(geo) if case.get("chart") else None
    eng = Engine(geo, chart=chart)
    s.update(geo=geo, tx=tx, ub=ub, ubn=ubn, engine=eng)
    if kind == "step":
        if case["path"] == "selector":
            eng.set_selector(Selector.load(MODEL_FILE), 0.9)
        elif case["path"] == "split":
            eng.set_precision(2)
        eng.set_targets(tx)
        eng.nearlist()
        s["far"] = eng.far(ub, ubn)
        s["u"] = np.zeros(eng.nt)
    return s


def run(s):
    kind = s["kind"]
    if kind == "closepanel":
        return rrq.lap3ddlp_closepanel(s["tx"], s["sx"], s["order"], ref=s["ref"])
    if kind == "rrq":
        r = rrq.rrq(s["tx"], s["sx"], s["snx"], s["sw"], s["rts"], s["rps"], s["order"], exterior=s["exterior"],
                    pre=s["pre"])
        return [r["As"], r["Ad"], r["Omega"], r["Ias"]]
    if kind == "getnearquad":
        return list(rrq.getnearquad_lap_rrq(s["geo"], s["tcx"], s["tcxrow"], s["tcxi"], iside=s["iside"]))
    if kind == "layer":
        return grf.layer_potential(s["geo"], s["tx"], s["ub"], s["ubn"], engine=s["engine"])[0]
    if kind == "mixed":
        return s["batch"].potential()
    eng = s["engine"]
    eng.set_potential(s["far"])
    eng.eval()
    eng.apply_resident()
    check(lib().qol_engine_get_values(eng._h, ctypes.c_void_p(), ptr(s["u"])), "qol_engine_get_values")
    return s["u"]


# ------------------------------------------------------------------ what it cannot do without
def _pair_work(p, pairs, panels):
    """flops and bytes of the close evaluation of `pairs` near pairs on `panels`
    panels of order p: level nodes, direct sums and their interpolation, RRQ
    moments and weights, one solve per panel; surface and targets in"""
    i = order_info(p)
    h, nb = i["h"], 3 * i["nq"]
    nc1, nc2, ncoef = p * (p + 1) // 2, p * (p - 1) // 2, i["ncoef"]
    direct = sum(f * int(n) * (19 + 4 * h) for f, n in zip(SHARES, i["nl"]))
    rrq_pair = 4 * nb * (3 * nc1 + 9 * nc2) + 400 * ncoef + 20 * h * h
    flops = pairs * (direct + SHARES[4] * rrq_pair) + panels * (18 * h * int(sum(i["nl"])) + 44 * h ** 3)
    return flops, 13 * 8 * panels * h + 24 * pairs / PAIRS_PER_TARGET


def work(case):
    kind, nt = case["kind"], case["targets"]
    if kind == "closepanel":
        # about four levels of cells, four leaves each, one q x q leaf rule a cell
        p, q = case["order"], 2 * case["order"] + 2 * case["ref"]
        return dict(flops=nt * 16.0 * q * q * (30 + 2 * p * p), bytes=8.0 * nt * (3 + p * p) + 24.0 * p * p)
    if kind == "rrq":
        h = case["order"] * (case["order"] + 1) // 2
        fl, by = _pair_work(case["order"], nt, 1)
        return dict(flops=fl, bytes=by + 8.0 * nt * (6 * h + 4))
    if kind == "mixed":
        surf = _mixed_surface(case["mp"], case["np"], tuple(int(p) for p in case["orders"].split(",")))
        fl = by = 0.0
        total = sum(g["ntri"] for g in surf["parts"].values())
        for p, g in surf["parts"].items():
            f, b = _pair_work(p, PAIRS_PER_TARGET * nt * g["ntri"] / total, g["ntri"])
            fl, by = fl + f, by + b
        return dict(flops=fl, bytes=by + 16.0 * nt)
    p = case["order"]
    geo = _surface(case["mp"], case["np"], p)
    npan, h = geo["ntri"], geo["h"]
    pairs = case["near"] * npan if kind == "getnearquad" else PAIRS_PER_TARGET * nt
    fl, by = _pair_work(p, pairs, npan)
    if kind == "getnearquad":
        return dict(flops=fl, bytes=by + 32.0 * pairs * h)
    if kind == "layer":
        fl += 26.0 * nt * npan * h
    return dict(flops=fl, bytes=by + 16.0 * npan * h + 16.0 * nt)


def exact(case, seed):
    """Green's identity: S[du/dn] - D[u] is u at the targets inside and 0 outside,
    the value that the layer potential approximates; None where a call returns
    weights, which have no closed form"""
    if case["kind"] not in ("layer", "step"):
        return None
    geo, tx, dist = _targets(case, seed)
    u, _ = W.charge_field(tx, *_charges(geo, seed + 2))
    return np.where(dist < 0.0, u, 0.0)
