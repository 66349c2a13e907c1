"""Transposed tree apply over leaf sizes at the edges of its output kernel: a
panel or two per leaf, more columns than one pass takes (16), more rows than
one list holds (512), more panels in a leaf than one slab (1024).  Each
layer is pinned against the forward apply by <y, A x> = <A^T y, x> (FP64 sums
of a few thousand terms: 1e-12 of the norms), FP32 against FP64 to 1e-5."""
import numpy as np
import pytest

import fftsvd_amd as fa
from fftsvd_amd import meshes

pytestmark = pytest.mark.gpu


def _dot(t, n, npt):
    rng = np.random.default_rng(n)
    y, x = rng.uniform(-1, 1, npt), rng.uniform(-1, 1, n)
    zero = np.zeros(n)
    for layer in (0, 1):
        fwd = t.apply_both(x, zero) if layer == 0 else t.apply_both(zero, x)
        adj = t.apply_transpose(layer, y)
        assert abs(y @ fwd - adj @ x) <= 1e-12 * np.linalg.norm(y) * np.linalg.norm(fwd)
        adj32 = t.apply_transpose(layer, y, fa.MIXED)
        assert np.linalg.norm(adj32 - adj) <= 1e-5 * np.linalg.norm(adj)


@pytest.mark.parametrize("sub,maxpanels,gridpoints", [(0, 32, 4), (2, 2, 4), (3, 17, 3), (3, 60, 4), (4, 200, 4), (3, 1300, 4)])
def test_transpose_against_forward(sub, maxpanels, gridpoints):
    V, F = meshes.ellipsoid((3.0, 2.2, 1.6), subdivisions=sub, jitter=0.04, seed=5)
    P = meshes.panels_from_mesh(V, F)
    g = fa.Problem(P, [[0.1, 0.2, -0.1]], [1.0], 4.0, 80.0, 0.124, maxpanels=maxpanels, gridpoints=gridpoints)
    for which in (0, 1):
        _dot(g.tree(which), len(P), len(P))
    # both layers at once, through the region operator
    rng = np.random.default_rng(1)
    x, y = rng.uniform(-1, 1, g.nvec), rng.uniform(-1, 1, g.nvec)
    for prec, tol in ((fa.F64, 1e-12), (fa.MIXED, 1e-5)):
        Ax = g.matvec(x, prec)
        assert abs(y @ Ax - g.matvec_transpose(y, prec) @ x) <= tol * np.linalg.norm(y) * np.linalg.norm(Ax)
