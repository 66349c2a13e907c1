"""The work that programs built on this framework have it do, as timed cases.

A program meshes a molecule (its solvent-excluded surface), builds the
compressed boundary-element operator, and then solves: one charge vector
(a solvation energy), many charge vectors on one operator, or a solve and
its gradients.  The cases are such passes through the Python entry points
(host arrays in and out), from one operator product on a small surface to
the whole calculation on about 100 000 panels.

The molecules are this repository's synthetic globules (a seeded
self-avoiding walk of atoms, its surface triangulated by the library's
mesher), Born spheres and jittered ellipsoids.  A molecule is fixed by the
case; the seed turns it to a random orientation (so the octree, the lists
and the operator are others) and draws its charges.

kinds
  matvec   operator products on host vectors (a program's own Krylov loop)
  solve    right-hand side, GMRES and potentials on an operator in hand
  whole    operator construction, right-hand side, GMRES, potentials
  batch    many charge vectors on an operator in hand
  gradq    gradient of the energy with respect to the charges
  gradk    derivative of the energy with respect to kappa
  qual     the second-kind (apparent surface charge) formulation, whole
  stern    the whole calculation with an ion-exclusion surface
"""
import functools
import math

import numpy as np
import torch

import fftsvd_amd as fa
from fftsvd_amd import meshes

EPS_IN, EPS_OUT, KAPPA = 4.0, 80.0, 0.124
TOL = 1e-6


def listed():
    return [
        # the smallest call: one product with a 1280-panel operator, FP64
        dict(name="matvec-1280-f64", kind="matvec", shape="ellipsoid", sub=3, mixed=False, kappa=KAPPA),
        # a program's own Krylov loop on a mid-size molecule, FP32 operator
        dict(name="matvec-30k-mixed", kind="matvec", shape="globule", atoms=500, spacing=1.27, mixed=True, kappa=KAPPA),
        # the Born ion, 5120 panels, no salt: GMRES on a small FP64 operator, bound by launches
        dict(name="solve-born5k-f64", kind="solve", shape="sphere", sub=4, mixed=False, kappa=0.0),
        # a further charge state of a large molecule on its operator, mixed precision
        dict(name="solve-100k-mixed", kind="solve", shape="globule", atoms=2000, spacing=1.266, mixed=True, kappa=KAPPA),
        # the same in FP64 on an ordinary molecule
        dict(name="solve-58k-f64", kind="solve", shape="globule", atoms=1000, spacing=1.31, mixed=False, kappa=KAPPA),
        # a small molecule from its panels to its potentials, as in a scan over many of them
        dict(name="whole-4k-mixed", kind="whole", shape="globule", atoms=60, spacing=1.27, mixed=True, kappa=KAPPA),
        # an ordinary molecule, FP64 only (the drop-in interface's default)
        dict(name="whole-30k-f64", kind="whole", shape="globule", atoms=500, spacing=1.27, mixed=False, kappa=KAPPA),
        # the whole calculation on the largest molecule, mixed precision
        dict(name="whole-100k-mixed", kind="whole", shape="globule", atoms=2000, spacing=1.266, mixed=True, kappa=KAPPA),
        # 64 charge vectors (a response matrix's columns) on one operator
        dict(name="batch64-30k-mixed", kind="batch", shape="globule", atoms=500, spacing=1.27, mixed=True, kappa=KAPPA,
             columns=64),
        # charge gradient after a solve (charge fitting)
        dict(name="gradq-30k-mixed", kind="gradq", shape="globule", atoms=500, spacing=1.27, mixed=True, kappa=KAPPA),
        # solveBEMproblem's settings: 27 panels a leaf, 3 grid points a side, GMRES to 1e-5
        dict(name="qual-18k-f64", kind="qual", shape="globule", atoms=250, spacing=1.25, mixed=False, kappa=0.0),
        # Stern layer: a salt surface around the molecule, three regions
        dict(name="stern-13k-mixed", kind="stern", shape="globule", atoms=200, spacing=1.3, mixed=True, kappa=KAPPA),
    ]


def draw(rng):
    kind = rng.choice(["matvec", "solve", "whole", "batch", "gradq", "gradk", "qual", "stern"])
    top = dict(matvec=1500, solve=1500, whole=1500, batch=300, gradq=700, gradk=700, qual=700, stern=400)[kind]
    c = dict(kind=kind, shape="globule", atoms=int(round(math.exp(rng.uniform(math.log(24), math.log(top))))),
             spacing=round(rng.uniform(1.2, 1.5), 3), mixed=rng.random() < 0.5, kappa=round(rng.uniform(0.04, 0.3), 3))
    if kind in ("solve", "whole") and rng.random() < 0.3 or kind == "qual":
        c["kappa"] = 0.0
    if kind == "batch":
        c["columns"] = rng.randint(2, 48)
    return c


# ---------------------------------------------------------------------------
# inputs


@functools.lru_cache(maxsize=8)
def _molecule(shape, size, spacing, stern):
    """(verts, faces, atom positions, salt surface verts and faces or None)."""
    if shape == "sphere":
        V, F = meshes.icosphere(2.0, size)
        return V, F, np.zeros((1, 3)), None, None
    if shape == "ellipsoid":
        V, F = meshes.ellipsoid((3.0, 2.2, 1.6), subdivisions=size, jitter=0.04, seed=7)
        return V, F, np.random.default_rng(1).uniform(-0.8, 0.8, size=(6, 3)), None, None
    xyz, radii, _ = meshes.synthetic_globule(natoms=size, seed=20261202)
    V, F = meshes.ses_mesh(xyz, radii, 1.4, spacing)
    if not stern:
        return V, F, xyz, None, None
    Vs, Fs = meshes.union_mesh(xyz, radii, 2.0, 1.3 * spacing)
    return V, F, xyz, Vs, Fs


def _base(case):
    return _molecule(case["shape"], case["atoms"] if case["shape"] == "globule" else case["sub"],
                     case.get("spacing", 0.0), case["kind"] == "stern")


def _inputs(case, seed):
    """Panels, charge positions, charges (and salt panels) of this seed."""
    V, F, xyz, Vs, Fs = _base(case)
    rng = np.random.default_rng(seed)
    Q, R = np.linalg.qr(rng.normal(size=(3, 3)))
    Q *= np.sign(np.diag(R))
    if np.linalg.det(Q) < 0:
        Q[:, 0] = -Q[:, 0]
    d = dict(panels=meshes.panels_from_mesh(V @ Q.T, F), qpos=np.ascontiguousarray(xyz @ Q.T))
    if Vs is not None:
        d["salt"] = meshes.panels_from_mesh(Vs @ Q.T, Fs)
    n = len(xyz)
    if n == 1:
        d["q"] = np.array([rng.uniform(0.5, 2.0)])
    else:
        q = rng.uniform(-0.8, 0.8, n)
        d["q"] = q + (np.round(q.sum()) - q.sum()) / n
    if case["kind"] == "batch":
        d["Q"] = np.asfortranarray(rng.uniform(-0.8, 0.8, size=(n, case["columns"])))
    if case["kind"] == "matvec":
        d["x"] = rng.uniform(-1.0, 1.0, 2 * len(d["panels"]))
    return d


def _problem(case, d):
    if case["kind"] == "qual":
        return fa.Qual(d["panels"], d["qpos"], d["q"], EPS_IN, EPS_OUT, maxpanels=27, gridpoints=3,
                       want_f32=case["mixed"])
    return fa.Problem(d["panels"], d["qpos"], d["q"], EPS_IN, EPS_OUT, case["kappa"], want_f32=case["mixed"],
                      stern_verts9=d.get("salt"))


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    kind = case["kind"]
    if kind in ("whole", "qual", "stern"):
        fa.lib()
        return s
    s["problem"] = p = _problem(case, s)
    s["prec"] = fa.MIXED if case["mixed"] else fa.F64
    if kind in ("gradq", "gradk"):
        s["solution"], _, _, _ = p.solve(p.rhs(), TOL, precision=s["prec"])
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    prec = fa.MIXED if case["mixed"] else fa.F64
    if kind == "matvec":
        return s["problem"].matvec(s["x"], prec)
    if kind == "solve":
        return _solve(s["problem"], prec, TOL)
    if kind == "batch":
        p = s["problem"]
        rhs = p.rhs_batch(s["Q"])
        sol, _, _ = p.solve_batch(rhs, TOL, precision=prec)
        return dict(rhs=rhs, solution=sol, potentials=p.potentials_batch(sol))
    if kind == "gradq":
        return s["problem"].grad_charges(s["solution"], TOL, precision=prec)
    if kind == "gradk":
        return s["problem"].grad_kappa(s["solution"], TOL, precision=prec)
    p = _problem(case, s)
    out = _solve(p, prec, 1e-5 if kind == "qual" else TOL)
    p.close()
    return out


def _solve(p, prec, tol):
    rhs = p.rhs()
    sol, _, _, _ = p.solve(rhs, tol, precision=prec)
    return dict(rhs=rhs, solution=sol, potentials=p.reaction_potentials(sol))


# ---------------------------------------------------------------------------
# what a pass cannot do without

# stored operator entries per unknown panel (near field, bases and their
# equivalent densities, both trees of a two-region operator), complex bins
# multiplied in its translations, and GMRES iterations to 1e-6, as these
# molecules have them
ENTRIES, MACS, ITERS = 2060.0, 3790.0, 85.0


def work(case):
    V, F, xyz, Vs, Fs = _base(case)
    n, nq = float(len(F)), float(len(xyz))
    if Fs is not None:
        n += 1.2 * len(Fs)
    kind = case["kind"]
    # one operator for the second-kind formulation
    share = 0.45 if kind == "qual" else 1.0
    size = 4.0 if case["mixed"] else 8.0
    nv = n if kind == "qual" else 2.0 * n
    mv_bytes, mv_flops = share * ENTRIES * size * n, share * (2.0 * ENTRIES + 8.0 * MACS) * n
    # a GMRES iteration: one product, the basis read and one vector written
    it = 12.0 if kind in ("qual",) or case["shape"] == "sphere" else ITERS
    sol_bytes = it * (mv_bytes + size * nv * it / 2.0)
    sol_flops = it * (mv_flops + 4.0 * nv * it / 2.0)
    # panel integrals at about 100 operations each
    pot = dict(bytes=656.0 * n + 8.0 * nv, flops=100.0 * n * nq)
    rhs_flops = 10.0 * n * nq
    if kind == "matvec":
        return dict(bytes=mv_bytes + 16.0 * nv, flops=mv_flops)
    if kind == "batch":
        m = float(case["columns"])
        return dict(bytes=it * mv_bytes + m * it * size * nv * it / 2.0 + pot["bytes"] + 32.0 * nv * m,
                    flops=m * sol_flops + pot["flops"] + m * 4.0 * n * nq)
    if kind == "gradq":
        return dict(bytes=sol_bytes + 2.0 * pot["bytes"], flops=sol_flops + 2.0 * pot["flops"] + rhs_flops)
    setup = dict(bytes=2.0 * share * ENTRIES * 8.0 * n, flops=3.0 * share * ENTRIES * 100.0 * n)
    if kind == "gradk":
        return dict(bytes=sol_bytes + setup["bytes"] + pot["bytes"], flops=sol_flops + setup["flops"] + pot["flops"])
    w = dict(bytes=sol_bytes + pot["bytes"] + 8.0 * nv, flops=sol_flops + pot["flops"] + rhs_flops)
    if kind in ("whole", "qual", "stern"):
        w = dict(bytes=w["bytes"] + setup["bytes"] + 72.0 * n, flops=w["flops"] + setup["flops"])
    return w


def tolerance(case):
    # About four times what the path shows against itself with other rounding
    # (the geometry scaled by one unit in the last place; FP32 against FP64
    # operators for a product).  A mixed solve's solution also moves by 1e-4
    # (3e-2 at its smallest entries) when its residual lands just on the other
    # side of the stopping test, one iteration sooner or later.
    kind, mixed = case["kind"], case["mixed"]
    if kind == "matvec":
        return dict(rel=6e-7, max=6e-6) if mixed else dict(rel=1e-13, max=1e-11)
    if not mixed:
        return dict(rel=1e-8, max=1e-5)
    if kind in ("gradq", "gradk"):
        return dict(rel=2e-6, max=7e-5)
    return dict(rel=2e-4, max=5e-2)


# ---------------------------------------------------------------------------
# the same in 64 bits: the dense operator with the panel integrals by
# Gauss-Legendre quadrature of their edge form

EXACT_PANELS = 5200


def _panel_frames(P):
    """Per panel: centroid, unit normal, vertices (n, 3, 3)."""
    v = P.reshape(-1, 3, 3)
    c = v.sum(1) / 3.0
    # the analytic normal of panel (v0, v1, v2) points along (v2-v0) x (v1-v0)
    nrm = torch.linalg.cross(v[:, 2] - v[:, 0], v[:, 1] - v[:, 0])
    return c, nrm / nrm.norm(dim=1, keepdim=True), v


def _integrals(pts, P, kappa):
    """Single and double layer of every panel at every point, (npt, npan).

    Over an edge at in-plane distance h (signed: positive towards the panel's
    inside) from the foot of the point, rho = h cosh u with u = asinh(t / h),
    d theta = du / cosh u; int dS e^{-kr}/r = sum over edges of
    int (e^{-k|z|} - e^{-kR}) / k d theta, R^2 = rho^2 + z^2."""
    c, nrm, v = _panel_frames(P)
    gx, gw = np.polynomial.legendre.leggauss(24)
    z = pts @ nrm.T - (c * nrm).sum(1)
    az = z.abs()
    S, D = torch.zeros_like(z), torch.zeros_like(z)
    self_ = ((pts[:, None, :] - c[None]).abs().amax(2) < 1e-12)
    ekz = torch.exp(-kappa * az)
    sgn = torch.where(z < 0, -1.0, 1.0).to(z)
    for j in range(3):
        a, b = v[:, j], v[:, (j + 1) % 3]
        e = (b - a) / (b - a).norm(dim=1, keepdim=True)
        m = torch.linalg.cross(e, nrm)     # in-plane, normal to the edge
        m = m * torch.sign(((a - c) * m).sum(1, keepdim=True))   # pointing out of the panel
        h = (a * m).sum(1) - pts @ m.T     # distance of the edge from the point's foot, outward
        t1, t2 = (a * e).sum(1) - pts @ e.T, (b * e).sum(1) - pts @ e.T
        ah = h.abs().clamp_min(1e-13)
        u1, u2 = torch.asinh(t1 / ah), torch.asinh(t2 / ah)
        um = torch.where((u1 < 0) & (u2 > 0), torch.zeros_like(u1), 0.5 * (u1 + u2))
        s, d = torch.zeros_like(z), torch.zeros_like(z)
        for lo, hi in ((u1, um), (um, u2)):
            half = 0.5 * (hi - lo)
            for x, w in zip(gx.tolist(), gw.tolist()):
                ch = torch.cosh(lo + half * (1.0 + x))
                R = torch.sqrt((ah * ch) ** 2 + z * z)
                wt = w * half / ch
                if kappa > 0:
                    ekr = torch.exp(-kappa * R)
                    s += wt * (ekz - ekr) / kappa
                    d += wt * (sgn * ekz - z / R * ekr)
                else:
                    s += wt * (R - az)
                    d += wt * (sgn - z / R)
        sg = torch.sign(h)
        S += sg * s
        D += sg * d
    flat = az < 1e-9
    D = torch.where(flat, torch.where(self_, 2.0 * math.pi, 0.0).to(D), D)
    return S, D


def _dense(P, kappa):
    """The 2N x 2N two-region operator and its right-hand-side rows."""
    c = _panel_frames(P)[0]
    n = len(P)
    A = torch.empty(2 * n, 2 * n, dtype=torch.float64, device=P.device)
    for i0 in range(0, n, 512):
        i1 = min(n, i0 + 512)
        S, D = _integrals(c[i0:i1], P, 0.0)
        A[i0:i1, :n], A[i0:i1, n:] = D, -S
        if kappa > 0:
            S, D = _integrals(c[i0:i1], P, kappa)
        A[n + i0:n + i1, :n], A[n + i0:n + i1, n:] = -D, EPS_IN / EPS_OUT * S
    k = torch.arange(n, device=P.device)
    A[n + k, k] += 4.0 * math.pi
    return A


def _coulomb(P, qpos):
    """1 / |charge - centroid|, (npan, ncharge)."""
    return 1.0 / torch.cdist(_panel_frames(P)[0], qpos, compute_mode="donot_use_mm_for_euclid_dist")


def exact(case, seed):
    kind = case["kind"]
    if kind == "gradk":
        return None
    d = _inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    P, qpos = (torch.as_tensor(d[k], dtype=torch.float64, device=dev) for k in ("panels", "qpos"))
    n = len(P)
    host = lambda t: np.ascontiguousarray(t.cpu().numpy())  # noqa: E731
    if kind == "qual":
        q = torch.as_tensor(d["q"], device=dev)
        rhs = torch.cat([-(_integrals(qpos, P[k:k + 2048], 0.0)[1].T @ q) for k in range(0, n, 2048)])
        return dict(rhs=host(rhs / (4.0 * math.pi * EPS_IN)), solution=None, potentials=None)
    if kind == "matvec":
        if n > EXACT_PANELS:
            return None
        return host(_dense(P, case["kappa"]) @ torch.as_tensor(d["x"], device=dev))
    q = torch.as_tensor(np.ascontiguousarray(d["Q"] if kind == "batch" else d["q"][:, None]), device=dev)
    B = _coulomb(P, qpos)
    top = B @ q
    rhs = torch.zeros(2 * n, q.shape[1], dtype=torch.float64, device=dev)
    rhs[:n] = top
    flat = (lambda t: np.asfortranarray(t.cpu().numpy())) if kind == "batch" else (lambda t: host(t[:, 0]))
    if kind == "stern":
        # the charges see the dielectric surface alone; its rows come after the salt surface's
        ns = len(d["salt"])
        full = np.zeros(2 * (ns + n))
        full[2 * ns:2 * ns + n] = host(top[:, 0])
        return dict(rhs=full, solution=None, potentials=None)
    if n > EXACT_PANELS:
        return None if kind == "gradq" else dict(rhs=flat(rhs), solution=None, potentials=None)
    A = _dense(P, case["kappa"])
    S, D = _integrals(qpos, P, 0.0)
    C = torch.cat([-D, S], 1)   # solution -> reaction potentials
    if kind == "gradq":
        q1 = q[:, 0]
        LU = torch.linalg.lu_factor(A)
        x = torch.linalg.lu_solve(*LU, rhs)
        lam = torch.linalg.lu_solve(*LU, (C.T @ q1)[:, None], adjoint=True)
        g = 0.5 * (C @ x[:, 0] + B.T @ lam[:n, 0])
        return host(g * 332.112 / EPS_IN)
    x = torch.linalg.solve(A, rhs)
    return dict(rhs=flat(rhs), solution=flat(x), potentials=flat(C @ x))
