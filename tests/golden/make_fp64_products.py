"""Writes fp64_products.json: sampled entries of FP64 operator products, the
fixture behind tests/test_gpu_fp64_products.py.  Needs the GPU.  The entries
were recorded with bases whose columns were written back at every step of the
pivoted MGS, one launch per step (the same order of every sum).

    python tests/golden/make_fp64_products.py
"""
import json
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
sys.path.insert(0, ROOT)

import fftsvd_amd as fa  # noqa: E402
from fftsvd_amd import meshes  # noqa: E402

# name: (surface, panels a leaf, SVD tolerance); the cubes' sampled matrices
# range over all kernels that make bases
CASES = {
    "leaves of 5": (("ellipsoid", 3), 5, 1e-5),
    "tight": (("ellipsoid", 3), 32, 1e-8),
    "leaves of 100": (("ellipsoid", 3), 100, 1e-6),
    "5120 panels": (("ellipsoid", 4), 70, 1e-5),
    "leaves of 300": (("ellipsoid", 4), 300, 1e-7),
    "20480 panels": (("ellipsoid", 5), 900, 1e-6),
    "81920 panels": (("ellipsoid", 6), 32, 1e-5),
    "two spheres": (("spheres", 5), 400, 1e-5),
    "globule": (("globule", 60), 32, 1e-5),
}


def panels(kind, size):
    if kind == "ellipsoid":
        return meshes.panels_from_mesh(*meshes.ellipsoid((3.0, 2.2, 1.6), subdivisions=size, jitter=0.04, seed=11))
    if kind == "spheres":   # each within one coarse cube
        V, F = meshes.icosphere(1.0, size)
        return np.vstack([meshes.panels_from_mesh(V, F), meshes.panels_from_mesh(V + 20.0, F)])
    xyz, radii, _ = meshes.synthetic_globule(natoms=size, seed=20261202)
    return meshes.panels_from_mesh(*meshes.ses_mesh(xyz, radii, 1.4, 1.27))


def product(name):
    """Norm and 48 entries of an FP64 product."""
    surface, maxpanels, svdeps = CASES[name]
    p = fa.Problem(panels(*surface), [[0.1, 0.2, -0.1]], [1.0], 4.0, 80.0, 0.124, maxpanels=maxpanels, svdeps=svdeps)
    y = p.matvec(np.random.default_rng(3).uniform(-1, 1, p.nvec), fa.F64)
    p.close()
    return float(np.linalg.norm(y)), y[np.random.default_rng(5).choice(len(y), 48, replace=False)]


if __name__ == "__main__":
    out = {}
    for name in CASES:
        norm, y = product(name)
        out[name] = dict(norm=norm.hex(), entries=[float(v).hex() for v in y])
        print(name, norm, flush=True)
    with open(sys.argv[1] if len(sys.argv) > 1 else os.path.join(HERE, "fp64_products.json"), "w") as f:
        json.dump(out, f, indent=0)
        f.write("\n")
