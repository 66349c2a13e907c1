"""Transposed tree apply over leaf sizes at the edges of its output kernel: a
panel or two per leaf, more columns than one pass takes (16), more rows than
one list holds (512), more panels in a leaf than one slab (1024).  Each
layer is pinned against the forward apply by <y, A x> = <A^T y, x> (FP64 sums
of a few thousand terms: 1e-12 of the norms), FP32 against FP64 to 1e-5."""
import ctypes as C

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


def test_each_precision_made_when_used():
    """The plan of one precision does not hold the point-major U of the other; the
    results do not depend on which came first."""
    V, F = meshes.ellipsoid((3.0, 2.2, 1.6), subdivisions=5, jitter=0.04, seed=5)
    P = meshes.panels_from_mesh(V, F)
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]

    def used():
        fa.release_memory()
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return t.value - f.value

    y = np.random.default_rng(2).uniform(-1, 1, 2 * len(P))
    out = {}
    for order in ((fa.MIXED, fa.F64), (fa.F64, fa.MIXED)):
        g = fa.Problem(P, [[0.1, 0.2, -0.1]], [1.0], 4.0, 80.0, 0.124)
        n_u = sum(c["colrank"] * c["npt"] for which in (0, 1) for c in g.tree(which).cubes())
        first = used()
        for prec in order:
            out[order, prec] = g.matvec_transpose(y, prec)
            now = used()
            assert now - first >= 0.9 * n_u * (8 if prec == fa.F64 else 4)
            first = now
        g.close()
    for prec in (fa.F64, fa.MIXED):
        np.testing.assert_array_equal(out[(fa.MIXED, fa.F64), prec], out[(fa.F64, fa.MIXED), prec])
