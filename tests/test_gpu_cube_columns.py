"""Far-field cubes of four grid points per side, one wavefront each: batches of
columns at the edges of their groups (four, two in FP64; two columns per
transform) equal the single product bit for bit; with trees whose cubes have
other sizes, one block each, beside them.  FP32 against FP64: 1e-5 (sums of a
few thousand 24-bit products)."""
import numpy as np
import pytest

import fftsvd_amd as fa
from fftsvd_amd import meshes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gridpoints,maxpanels", [(4, 8), (4, 40), (3, 12)])
def test_columns(gridpoints, maxpanels):
    V, F = meshes.ellipsoid((3.0, 2.2, 1.6), subdivisions=3, jitter=0.04, seed=3)
    P = meshes.panels_from_mesh(V, F)
    g = fa.Problem(P, [[0.1, 0.2, -0.1]], [1.0], 4.0, 80.0, 0.124, maxpanels=maxpanels, gridpoints=gridpoints)
    X = np.random.default_rng(gridpoints).uniform(-1, 1, (g.nvec, 7))
    single = {}
    for prec in (fa.F64, fa.MIXED):
        single[prec] = np.stack([g.matvec(X[:, c], prec) for c in range(7)], axis=1)
        for ncol in (2, 3, 4, 5, 7):
            np.testing.assert_array_equal(g.matvec_batch(X[:, :ncol], prec), single[prec][:, :ncol])
    assert np.linalg.norm(single[fa.MIXED] - single[fa.F64]) <= 1e-5 * np.linalg.norm(single[fa.F64])
    g.close()
