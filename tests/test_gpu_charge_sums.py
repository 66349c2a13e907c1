"""Charge right-hand sides and reaction potentials against plain sums over
charges and panels, at charge counts around a wave's 64 lanes, panel counts
around a block's 256 and column counts around one pass (8, 16, 32, 64).  FP64
sums in another order: 1e-13 of the sum of absolute values; the panel integrals
are the library's own, one pair at a time.  A charge on a centroid with value
zero adds nothing to the right-hand side.

Their transposes (collection and right-hand side) through the charge gradient
1/2 (C x + B^T lambda), A^T lambda = C^T q, with plain sums for C and B, at charge
counts around one part of the walk over charges (16) and a wave's lanes.  The
adjoint solve to 1e-12 of its right-hand side lies between: 1e-9."""
import numpy as np
import pytest

import fftsvd_amd as fa
import oracle
from fftsvd_amd import meshes

pytestmark = pytest.mark.gpu
AXES = np.array([6.0, 5.0, 4.0])


def _problem(sub, nq):
    V, F = meshes.ellipsoid(tuple(AXES), subdivisions=sub, jitter=0.04, seed=sub)
    P = meshes.panels_from_mesh(V, F)
    rng = np.random.default_rng(nq)
    x = rng.normal(size=(nq, 3))
    x *= AXES * 0.97 * rng.uniform(0, 1, (nq, 1)) ** (1 / 3) / np.linalg.norm(x, axis=1)[:, None]
    return P, x, rng


@pytest.mark.parametrize("sub,nq", [(1, 1), (1, 63), (2, 64), (2, 65), (3, 1), (3, 300)])
@pytest.mark.parametrize("ncol", [1, 3, 17, 65])
def test_sums(sub, nq, ncol):
    P, x, rng = _problem(sub, nq)
    n = len(P)
    q = rng.uniform(-1, 1, nq)
    g = fa.Problem(P, x, q, 4.0, 80.0, 0.124)
    cent = P.reshape(n, 3, 3).mean(axis=1)
    w = 1.0 / np.linalg.norm(x[None] - cent[:, None], axis=2)
    rhs = g.rhs()
    assert np.all(np.abs(rhs[:n] - w @ q) <= 1e-13 * (w @ np.abs(q)))
    Q = rng.uniform(-1, 1, (nq, ncol))
    R = g.rhs_batch(Q)
    assert np.all(np.abs(R[:n] - w @ Q) <= 1e-13 * (w @ np.abs(Q)))
    sl, dl = fa.integrate(P, x)
    S = rng.uniform(-1, 1, (g.nvec, ncol))
    ref, mag = sl @ S[n:] - dl @ S[:n], np.abs(sl) @ np.abs(S[n:]) + np.abs(dl) @ np.abs(S[:n])
    phi = g.potentials_batch(S)
    assert np.all(np.abs(phi - ref) <= 1e-13 * mag)
    for c in {0, ncol - 1}:
        assert np.all(np.abs(g.reaction_potentials(S[:, c]) - ref[:, c]) <= 1e-13 * mag[:, c])
    g.close()


def test_zero_charge_on_a_centroid():
    P, x, rng = _problem(2, 70)
    x[7] = P[11].reshape(3, 3).mean(axis=0)
    q = rng.uniform(-1, 1, 70)
    q[7] = 0.0
    keep = np.arange(70) != 7
    g, h = (fa.Problem(P, x[k], q[k], 4.0, 80.0, 0.124) for k in (slice(None), keep))
    R = g.rhs_batch(np.stack([q, -q], axis=1))
    for r in (g.rhs(), R[:, 0], -R[:, 1]):
        assert np.linalg.norm(r - h.rhs()) <= 1e-13 * np.linalg.norm(r)


@pytest.mark.parametrize("nq", [1, 16, 17, 63, 64, 65, 300])
@pytest.mark.parametrize("centroid", [False, True])
def test_transposes(nq, centroid):
    P, x, rng = _problem(2, nq)
    n = len(P)
    cent = P.reshape(n, 3, 3).mean(axis=1)
    if centroid:   # the charge's own gradient is infinite, the others see its 4 pi term
        x[nq // 2] = oracle.panel_geom(P[11])["centroid"]
    q = rng.uniform(-1, 1, nq)
    g = fa.Problem(P, x, q, 4.0, 80.0, 0.124)
    sl, dl = fa.integrate(P, x)
    if centroid:
        dl[nq // 2, 11] += 4.0 * np.pi
    C = np.hstack([-dl, sl])
    sol = rng.uniform(-1, 1, g.nvec)
    lam, _ = g.solve_adjoint(C.T @ q, 1e-12)
    grad = g.grad_charges(sol, 1e-12, conversion=g.eps_in)
    for j in range(nq):
        if centroid and j == nq // 2:
            continue
        w = 1.0 / np.linalg.norm(x[j] - cent, axis=1)
        ref, mag = 0.5 * (C[j] @ sol + w @ lam[:n]), np.abs(C[j]) @ np.abs(sol) + w @ np.abs(lam[:n])
        assert abs(grad[j] - ref) <= 1e-9 * mag
    g.close()


@pytest.mark.parametrize("sub,nq", [(1, 5), (3, 65)])
def test_qualocation(sub, nq):
    P, x, rng = _problem(sub, nq)
    q = rng.uniform(-1, 1, nq)
    g = fa.Qual(P, x, q, 4.0, 80.0)
    sl, dl = fa.integrate(P, x)
    f = -1.0 / (16.0 * np.pi)
    assert np.all(np.abs(g.rhs() - f * (dl.T @ q)) <= 1e-13 * abs(f) * (np.abs(dl).T @ np.abs(q)))
    s = rng.uniform(-1, 1, len(P))
    assert np.all(np.abs(g.potentials(s) - sl @ s) <= 1e-13 * (np.abs(sl) @ np.abs(s)))
