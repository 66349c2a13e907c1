"""Sampled column and row bases (pivoted MGS) over the sizes that their kernels
take: ranks equal to the oracle's for leaf sizes and SVD tolerances that reach a
lane per column (rows in registers, and beyond them in LDS), two columns a lane
group, the blocked kernel, and the one for the longest columns (cubes of 20480
panels); bases orthonormal to the level that pivoted MGS keeps, eps / svdeps
times a factor for the sums.  Their rounding: tests/test_gpu_fp64_products.py."""
import numpy as np
import pytest

import fftsvd_amd as fa
import oracle
from fftsvd_amd import meshes
from test_gpu_parity import _key

pytestmark = pytest.mark.gpu


def _bases(t, c):
    """VT (r x np) and U (nq x r') of a cube, its other blocks unread."""
    m = len(c["dcols"])
    VT, U = np.zeros(max(c["rowrank"] * c["npan"], 1)), np.zeros(max(c["npt"] * c["colrank"], 1))
    gp3 = 729
    PVs, PVd, UTI = (np.zeros(max(gp3 * r, 1)) for r in (c["rowrank"], c["rowrank"], c["colrank"]))
    Ds, Dd = np.zeros(max(c["npt"] * m, 1)), np.zeros(max(c["npt"] * m, 1))
    fa._check(fa.lib().fftsvd_tree_cube_mats(t.p.h, t.which, c["id"], *(fa._d(a) for a in (VT, U, PVs, PVd, UTI, Ds, Dd))))
    return (VT[:c["rowrank"] * c["npan"]].reshape(c["rowrank"], c["npan"]),
            U[:c["npt"] * c["colrank"]].reshape(c["npt"], c["colrank"]))


def _orthonormality(t, cubes):
    worst = 0.0
    for c in cubes:
        VT, U = _bases(t, c)
        for B in (VT, U.T):
            if len(B):
                worst = max(worst, np.abs(B @ B.T - np.eye(len(B))).max())
    return worst


@pytest.mark.parametrize("sub,maxpanels,svdeps", [(3, 5, 1e-5), (3, 32, 1e-8), (3, 100, 1e-6), (4, 70, 1e-5),
                                                  (4, 300, 1e-7)])
def test_ranks_match_oracle(sub, maxpanels, svdeps):
    V, F = meshes.ellipsoid((3.0, 2.2, 1.6), subdivisions=sub, jitter=0.04, seed=11)
    P = meshes.panels_from_mesh(V, F)
    args = (P, [[0.1, 0.2, -0.1]], [1.0], 4.0, 80.0, 0.124)
    g = fa.Problem(*args, maxpanels=maxpanels, svdeps=svdeps)
    o = oracle.Problem(*args, maxpanels=maxpanels, svdeps=svdeps)
    for which in (0, 1):
        gt, ot = g.tree(which), o.tree(which)
        gc = {_key(c): c for c in gt.cubes()}
        oc = {_key(c): c for c in ot.cubes()}
        assert set(gc) == set(oc)
        assert [(gc[k]["rowrank"], gc[k]["colrank"]) for k in oc] == [(c["rowrank"], c["colrank"]) for c in oc.values()]
        # 100 sums of eps, amplified by the smallest kept pivot svdeps
        assert _orthonormality(gt, gc.values()) <= 100 * 2.3e-16 / svdeps


def test_cubes_beyond_lds():
    # two spheres of 20480 panels, each within one level-2 cube
    V, F = meshes.icosphere(1.0, 5)
    P1 = meshes.panels_from_mesh(V, F)
    P2 = meshes.panels_from_mesh(V + 20.0, F)
    g = fa.Problem(np.vstack([P1, P2]), [[0.1, 0.2, -0.1]], [1.0], 4.0, 80.0, 0.0, maxpanels=400)
    t = g.tree(0)
    big = [c for c in t.cubes() if c["level"] == 2 and c["rowrank"] > 0]
    assert len(big) == 2 and all(c["npan"] == 20480 for c in big)
    assert _orthonormality(t, big) <= 100 * 2.3e-16 / 1e-5
    # the spheres see each other through these bases alone
    n = len(P1)
    rng = np.random.default_rng(3)
    xs, xd = np.zeros(2 * n), np.zeros(2 * n)
    xs[n:], xd[n:] = rng.uniform(0, 1, n), rng.uniform(-1, 1, n)
    y = t.apply_both(xs, xd)
    at = rng.choice(n, 40, replace=False)
    s, d = fa.integrate(P2, P1.reshape(-1, 3, 3)[at].mean(1))
    ref = s @ xs[n:] + d @ xd[n:]
    assert np.abs(y[at] - ref).max() <= 1e-4 * np.abs(ref).max()
