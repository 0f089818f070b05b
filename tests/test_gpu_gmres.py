"""The mixed solver's GMRES (device-resident Arnoldi steps) against the FP64
BiCG solution: vectors shorter than a reduction chunk, with remainders, with a
restart (more than 120 steps), and with an iteration limit.

At |r|^2/|b|^2 < 1e-14 both solutions carry a relative residual of 1e-7; their
difference is that times the condition of A, below 1e2 for the ordinary
clusters (1e-5) and below 1e3 for the resonant one (1e-4)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(ctx, n, x, ri, fv, solver, **kw):
    from mstm_amd import geometry as G

    c = G.rsa_in_sphere(n, x, fv, seed=7, ri=ri)
    ctx.set_spheres(c.pos, c.radius, c.ri, 1.0, 1e-6)
    return ctx.fixedorsoln(alpha=0.3, sinc=0.5, solver=solver, **kw)


@pytest.mark.parametrize("n,x,ri,fv,tol,restart", [(2, 0.5, 1.5 + 0.01j, 0.05, 1e-5, False),
                                                   (3, 1.0, 1.5 + 0.01j, 0.1, 1e-5, False),
                                                   (67, 1.5, 1.4 + 0.0j, 0.2, 1e-5, False),
                                                   (300, 2.5, 1.9 + 0.0j, 0.3, 1e-4, True)])
def test_mixed_gmres_matches_fp64(gpu_ctx, n, x, ri, fv, tol, restart):
    from mstm_amd.solver import SOLVE_MIXED, SOLVE_PLAIN

    ref = _solve(gpu_ctx, n, x, ri, fv, SOLVE_PLAIN, eps=1e-14)
    gpu_ctx.clear(clear_tables=False)
    r = _solve(gpu_ctx, n, x, ri, fv, SOLVE_MIXED, eps=1e-14)
    st = gpu_ctx.stats()
    assert r["maxerr"] < 1e-14 and r["istat"] == 0
    assert np.abs(r["amnp"] - ref["amnp"]).max() <= tol * np.abs(ref["amnp"]).max()
    if restart:
        assert st["iters_fp32"] > 2 * 120
    # repeated solves give the same bits
    again = _solve(gpu_ctx, n, x, ri, fv, SOLVE_MIXED, eps=1e-14)
    assert np.array_equal(again["amnp"], r["amnp"])


def test_mixed_gmres_iteration_limit(gpu_ctx):
    """A limit below what the solve needs: the count stops at it, and the
    products are counted as made."""
    from mstm_amd.solver import SOLVE_MIXED

    _solve(gpu_ctx, 67, 1.5, 1.4 + 0.0j, 0.2, SOLVE_MIXED, eps=1e-14, niter=1)  # tables
    gpu_ctx.clear(clear_tables=False)
    r = _solve(gpu_ctx, 67, 1.5, 1.4 + 0.0j, 0.2, SOLVE_MIXED, eps=1e-14, niter=5)
    st = gpu_ctx.stats()
    assert r["istat"] == 1 and r["iterations"] >= 5
    assert st["matvecs_fp32"] == 5 and st["iters_fp32"] == 10


def test_mixed_falls_back_when_fp32_overflows(gpu_ctx):
    """Two touching grains of x = 1e-4 beside a sphere of order 8: at the common
    order their table's row of degree 1 holds h_9(2e-4), about 3e44, above the
    FP32 range, and its product with the grains' zero padding is NaN.  The mixed
    solver ends its inner solves and answers with FP64 BiCG."""
    from mstm_amd.solver import FP32, SOLVE_MIXED, SOLVE_PLAIN

    pos = np.array([[0.0, 0.0, 0.0], [4.65, 0.0, 0.0], [4.65, 2e-4, 0.0], [0.0, 0.0, 12.0]])
    gpu_ctx.set_spheres(pos, np.array([4.6, 1e-4, 1e-4, 4.0]), np.full(4, 1.4 + 0.01j), 1.0, 1e-6)
    assert gpu_ctx.orders()[0].max() == 8
    one = np.ones((1, gpu_ctx.number_eqns), complex)
    assert np.isnan(gpu_ctx.sphereinteraction(one, [False], [True], precision=FP32)).any()
    ref = gpu_ctx.fixedorsoln(alpha=0.3, sinc=0.5, solver=SOLVE_PLAIN, eps=1e-14)
    gpu_ctx.clear(clear_tables=False)
    r = gpu_ctx.fixedorsoln(alpha=0.3, sinc=0.5, solver=SOLVE_MIXED, eps=1e-14)
    st = gpu_ctx.stats()
    assert r["istat"] == 0 and r["maxerr"] < 1e-14 and st["lig_fallbacks"] == 2
    assert np.abs(r["amnp"] - ref["amnp"]).max() <= 1e-5 * np.abs(ref["amnp"]).max()
