"""qol_lap3ddlp_closepanel_mex_ (tensor-patch close DLP, a15) on the GPU
against the oracle, the flat-square solid angle, and the reference's own
smoke test test/test_lap3d_close.f90 compiled unchanged against the Fortran
modules (oracle/_ref/test_lap3d_close, built by oracle/fortran_bench.mk)."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

from qotential_amd import rrq as R
from test_oracle_closepanel import _solid_square, flat_square, torus_patch

pytestmark = pytest.mark.gpu
BUILT = Path(__file__).resolve().parents[1] / "oracle" / "_ref" / "test_lap3d_close"


def test_closepanel_gpu_vs_oracle(oracle):
    print("tensor-patch close DLP: torus patch order 8 and flat square order 6", flush=True)
    p = 8
    sx = torus_patch(oracle, p)
    rng = np.random.default_rng(2)
    n = np.array([0.0, 0.0, 1.0])
    xs = np.vstack([[[0.05 * k, 0.03 * k - 0.05, 0.02 * k + 0.01] for k in range(1, 6)],
                    sx[rng.integers(0, p * p, 6)] + (10.0 ** rng.uniform(-7, -1, 6) * rng.choice([-1, 1], 6))[:, None] * n])
    g = R.lap3ddlp_closepanel(xs, sx, p)
    o = oracle.closepanel_dlp(xs, sx, p)
    rel = np.abs(g - o).max(1) / np.abs(o).max(1)
    print("max rel diff per row", rel.max(), flush=True)
    assert rel.max() < 1e-9  # the two quadtrees may split a cell differently at a rounding boundary
    ps, a = 6, 0.1
    sq = flat_square(oracle, ps, a)
    xq = np.array([[0.01, 0.02, 0.05], [0.0, 0.0, 1e-6], [0.099, -0.02, 2e-5]])
    gq = R.lap3ddlp_closepanel(xq, sq, ps)
    for i, x in enumerate(xq):
        assert abs(gq[i].sum() + _solid_square(x, a) / (4 * np.pi)) < 2e-11
    with pytest.raises(Exception, match="if_adapt"):
        R.lap3ddlp_closepanel(xq, sq, ps, if_adapt=False)


@pytest.mark.skipif(not BUILT.exists(), reason="oracle/_ref/test_lap3d_close not built (no reference checkout)")
def test_reference_smoke_test_runs():
    r = subprocess.run([str(BUILT)], capture_output=True, text=True, timeout=300)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0 and "PASS" in r.stdout


@pytest.mark.parametrize("p,ref,m", [(2, 1, 1), (3, 1, 205), (5, 11, 3), (5, 12, 2), (5, 18, 2), (7, 1, 40), (16, 1, 2)])
def test_closepanel_orders_and_blocks(oracle, p, ref, m):
    """the smallest and largest order, rules of one and of several blocks of
    nodes (q = 32, 34, 46), one and several parts per target; the bound is the
    one above (a cell's split test may fall differently)"""
    sx = torus_patch(oracle, p)
    rng = np.random.default_rng(p + ref + m)
    lo = -5 if p < 16 else -1.5
    xs = sx[rng.integers(0, p * p, m)] + (10.0 ** rng.uniform(lo, -1, m) * rng.choice([-1, 1], m))[:, None] * np.array([0.0, 0.0, 1.0])
    g = R.lap3ddlp_closepanel(xs, sx, p, ref=ref)
    pick = np.unique(np.concatenate([[0, m - 1], rng.integers(0, m, 6)]))
    o = oracle.closepanel_dlp(xs[pick], sx, p, ref=ref)
    rel = np.abs(g[pick] - o).max(1) / np.abs(o).max(1)
    print(p, ref, m, "max rel diff per row", rel.max(), flush=True)
    assert rel.max() < 1e-9
    assert np.array_equal(g, R.lap3ddlp_closepanel(xs, sx, p, ref=ref))


def test_closepanel_tree_limit(oracle):
    sx = torus_patch(oracle, 6)
    xs = np.array([[0.0, 0.0, 0.3], sx[14]])  # the second lies on the patch: its tree has no end
    far = R.lap3ddlp_closepanel(np.array([[0.0, 1e160, 0.0]]), sx, 6)
    assert np.all(far == 0.0)  # r^2 overflows
    with pytest.raises(Exception, match="size limit"):
        R.lap3ddlp_closepanel(xs, sx, 6)
