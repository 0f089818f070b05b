"""The mixed solver's GMRES decisions (gmres.hpp) without a GPU: cycles,
restarts and limits on small dense systems, and products that overflow.  A
product that is not finite ends the solve at once, with the correction of the
steps before it and an error above eps (the callers then solve in FP64)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def gmres(tmp_path_factory):
    from mstm_amd.build import HIPCC

    so = str(tmp_path_factory.mktemp("gmres") / "gmres_host.so")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-shared",
                    os.path.join(HERE, "native", "gmres_host.cpp"), "-o", so], check=True)
    fn = C.CDLL(so).gmres_host
    fn.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_double, C.c_int, C.c_int, C.c_int, C.c_double, C.c_int,
                   C.c_void_p, C.c_void_p]

    def solve(A, b, eps, niter, m, bad=10 ** 9, poison=0.0):
        x, out = np.zeros(len(b), complex), np.zeros(3)
        A = np.ascontiguousarray(A)
        closed = fn(len(b), A.ctypes.data, b.ctypes.data, eps, niter, m, bad, poison, 200, x.ctypes.data,
                    out.ctypes.data) == 0
        return x, int(out[0]), out[1], int(out[2]), closed

    return solve


def _system(n=24):
    rng = np.random.default_rng(5)
    A = np.eye(n) + 0.4 / np.sqrt(n) * (rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n)))
    return A, rng.normal(size=n) + 1j * rng.normal(size=n)


@pytest.mark.parametrize("m", [3, 7, 120])
def test_solves_across_restarts(gmres, m):
    A, b = _system()
    x, it, err, cycles, closed = gmres(A, b, 1e-20, 1000, m)
    assert closed and err < 1e-20 and cycles == -(-it // m)
    # relative residual 1e-10 times the condition of A (below 10)
    assert np.abs(x - np.linalg.solve(A, b)).max() <= 1e-9 * np.abs(x).max()


def test_iteration_limit(gmres):
    A, b = _system()
    x, it, err, cycles, closed = gmres(A, b, 1e-30, 5, 3)
    assert closed and it == 5 and err > 1e-30


@pytest.mark.parametrize("poison", [np.nan, np.inf, -np.inf, 1e200])
@pytest.mark.parametrize("bad", [0, 1, 4, 7, 8, 9])
def test_products_that_overflow_end_the_solve(gmres, bad, poison):
    """m = 7: product 7 is the second cycle's residual."""
    A, b = _system()
    x, it, err, cycles, closed = gmres(A, b, 1e-20, 10000, 7, bad, poison)
    assert closed
    assert np.isfinite(x).all() and err >= 1e-20
    if poison != 1e200:
        # what the finite steps gave
        ok = min(bad, 7) if bad <= 7 else bad - 1
        assert it == ok
        y, _, _, _, _ = gmres(A, b, 1e-30, ok, 7) if ok else (np.zeros_like(x),) * 5
        assert np.abs(x - y).max() <= 1e-12 * max(1.0, np.abs(y).max())
    assert np.linalg.norm(b - A @ x) <= np.linalg.norm(b) * (1 + 1e-12)


@pytest.mark.parametrize("bb", [np.nan, np.inf])
def test_right_hand_side_that_is_not_finite(gmres, bb):
    A, b = _system()
    b[3] = bb
    x, it, err, cycles, closed = gmres(A, b, 1e-20, 10000, 7)
    assert closed and it == 0 and not x.any()
