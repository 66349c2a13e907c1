"""Kept device memory (devmem.cpp): problems built, used and destroyed in turn
and on several threads at once, in blocks that earlier ones gave back, give the
same bits, also where every block is filled with NaN before it is handed out;
memory kept from a large problem goes back to the device once later builds have
not taken it, or when it is asked for."""
import ctypes as C
import os
import threading

import numpy as np
import pytest

import fftsvd_amd as fa
from fftsvd_amd import meshes

pytestmark = pytest.mark.gpu


def _pass(sub, kappa):
    V, F = meshes.ellipsoid((3.0, 2.2, 1.6), subdivisions=sub, jitter=0.04, seed=7)
    p = fa.Problem(meshes.panels_from_mesh(V, F), [[0.1, 0.2, -0.1], [-0.5, 0.1, 0.3]], [1.0, -0.4], 4.0, 80.0, kappa)
    x = np.random.default_rng(sub).uniform(-1, 1, p.nvec)
    sol, _, _, _ = p.solve(p.rhs(), precision=fa.MIXED)
    out = [p.matvec(x, fa.F64), p.matvec(x, fa.MIXED), sol, p.reaction_potentials(sol)]
    p.close()
    return out


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("threads", [1, 4])
def test_reused_blocks_same_results(threads):
    cases = [(2, 0.124), (3, 0.0), (3, 0.124), (4, 0.2)]
    first = [_pass(*c) for c in cases]
    bad = []

    def work(t):
        for k in range(4):
            i = (t + k) % len(cases)
            if not _same(_pass(*cases[i]), first[i]):
                bad.append((t, i))

    th = [threading.Thread(target=work, args=(t,)) for t in range(threads)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad


@pytest.mark.parametrize("threads", [1, 3])
def test_filled_blocks_same_results(threads):
    cases = [(2, 0.124), (3, 0.0), (4, 0.2)]
    first = [_pass(*c) for c in cases]
    got = {}
    os.environ["FFTSVD_FILL_MEMORY"] = "1"
    try:
        th = [threading.Thread(target=lambda t=t: got.update({t: [_pass(*c) for c in cases]})) for t in range(threads)]
        for t in th:
            t.start()
        for t in th:
            t.join()
    finally:
        del os.environ["FFTSVD_FILL_MEMORY"]
    for t in range(threads):
        assert all(_same(a, b) for a, b in zip(got[t], first))


def _memory():
    fa.lib()
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
    f, t = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value, t.value


def _free():
    return _memory()[0]


def test_kept_memory_goes_back():
    for _ in range(4):
        _pass(2, 0.124)
    base, total = _memory()
    _pass(5, 0.124)   # 20480 panels: more than 1 GB
    kept = base - _free()
    assert 512 << 20 < kept <= total // 24 + (64 << 20)
    for _ in range(4):
        _pass(2, 0.124)
    assert base - _free() <= 256 << 20


def test_release_memory():
    _pass(4, 0.124)
    before = _free()
    n = fa.release_memory()
    assert n > 128 << 20
    # blocks are whole pages for the runtime
    assert _free() - before >= n // 2
    assert fa.release_memory() == 0
