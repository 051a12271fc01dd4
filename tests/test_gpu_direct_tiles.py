"""The direct level kernel's tiles of 16 pairs against numpy on the engine's own
level nodes: tiles of one panel, of 4, 5, 8 and 16 panels (three chunk forms), a
last tile with dead lanes, every remainder of the column count, on every level."""
import numpy as np
import pytest

from qotential_amd import workload as W
from qotential_amd.engine import Engine, order_level

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12])
@pytest.mark.parametrize("per", [1, 2, 3, 4, 17])
def test_direct_tiles_vs_numpy(p, per):
    geo = W.geometry(4, 8, p, modes=W.VMEC_BENCH)
    npan = geo["ntri"]
    e = Engine(geo)
    cnt = np.where(np.arange(npan) < 19, per, 0)
    offs = np.concatenate([[0], np.cumsum(cnt)])
    tx = W.targets(geo, int(offs[-1]), -2.0, 0.0, sides=0, seed=p)[0]
    tx[1] = 0.5  # far off
    e.set_targets(tx)
    e.set_pairs(offs, 1 + np.arange(offs[-1]))
    info = e.level_info()
    lg, _ = e.level_data()
    panel = np.repeat(np.arange(npan), cnt)
    first = np.concatenate([[0], np.cumsum(info["nl"])])
    for lev in (1, 2, 3, 4):
        e.force_label(lev)
        e.eval()
        w = e.weights()
        im = order_level(p, lev)["interpmat"]
        g = lg[panel][:, :, first[lev - 1]:first[lev]]  # pairs, 7, nodes
        d = tx[:, :, None] - g[:, :3]
        r = np.sqrt((d * d).sum(1))
        s = g[:, 6] / (4 * np.pi * r)
        dk = s * (d * g[:, 3:6]).sum(1) / r ** 2
        for key, k, mag in (("As", s, s), ("Ad", dk, s / r)):
            ref, bound = k @ im, mag @ np.abs(im)
            err = np.abs(w[key] - ref) / bound
            # entries to 16 roundings, sums of n products on both sides
            assert err.max() <= (2 * im.shape[0] + 16) * 1.2e-16, (p, per, lev, key, err.max())


@pytest.mark.parametrize("p", [4, 6])
def test_many_tiles_vs_numpy(p):
    """enough pairs that one wave takes a tile (the lists above are short: four
    share one), in tiles of 1 to 16 panels"""
    geo = W.geometry(48, 120, p, modes=W.VMEC_BENCH)
    npan, h = geo["ntri"], geo["h"]
    cnt = np.where(np.arange(npan) % 1000 < 700, 1, 2)
    cnt[:3000] = 5
    cnt[3000:5000] = 121
    offs = np.concatenate([[0], np.cumsum(cnt)])
    n = int(offs[-1])
    assert n > 16 * 16384
    tx = W.targets(geo, n, -1.0, 0.0, sides=0, seed=p)[0]
    e = Engine(geo)
    e.set_targets(tx)
    e.set_pairs(offs, 1 + np.arange(n))
    panel = np.repeat(np.arange(npan), cnt)
    pick = np.concatenate([np.arange(40), n - 1 - np.arange(20), np.random.default_rng(p).integers(0, n, 140)])
    for lev in (1, 4):
        e.force_label(lev)
        e.eval()
        w = e.weights()
        lv = order_level(p, lev)
        im = lv["interpmat"]
        for j in pick:
            rows = slice(panel[j] * h, (panel[j] + 1) * h)
            x, xu, xv = im @ geo["sx"][rows], im @ geo["rts"][rows], im @ geo["rps"][rows]
            nn = np.cross(xv, xu)  # the normal as the level kernel forms it
            sp = np.linalg.norm(nn, axis=1)
            d = tx[j] - x
            r = np.linalg.norm(d, axis=1)
            s = sp * lv["wt"] / (4 * np.pi * r)
            k = s * (d * nn / sp[:, None]).sum(1) / r ** 2
            for key, v, mag in (("As", s, s), ("Ad", k, s / r)):
                # the nodes of both sides agree to 1e-15 of |x| ~ 1, at least 1e-3 from the target
                assert np.abs(w[key][j] - v @ im).max() <= 1e-11 * (mag @ np.abs(im)).max(), (lev, j, key)
