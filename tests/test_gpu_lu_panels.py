"""LU solutions whose panels end at the edges of the factorization's blocks: one
short panel, full workgroups and panels, remainders of 256 rows and 32 columns,
spheres of unequal order, 28 and all 64 workgroups.

The BiCG solution at |r|^2/|b|^2 < 1e-20 carries a relative residual of 1e-10;
times a condition below 1e2 that is 1e-8, taken ten times wider."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,x,spread,neq", [(1, 0.05, 0.0, None), (16, 1.0, 0.0, 768), (17, 0.3, 0.0, 510),
                                            (9, 0.3, 0.0, 270), (33, 0.9, 0.7, None), (100, 2.0, 0.0, 7000),
                                            (234, 2.0, 0.0, 16380)])
def test_lu_matches_bicg(gpu_ctx, n, x, spread, neq):
    from mstm_amd import geometry as G
    from mstm_amd.solver import SOLVE_LU, SOLVE_PLAIN

    c = G.rsa_in_sphere(n, x, 0.15, seed=3, ri=1.31 + 0.01j)
    radius = c.radius.copy()
    radius[1::3] *= 1.0 - spread
    gpu_ctx.set_spheres(c.pos, radius, c.ri, 1.0, 1e-6)
    if neq:
        assert gpu_ctx.number_eqns == neq
    r = gpu_ctx.fixedorsoln(alpha=0.4, sinc=0.3, solver=SOLVE_LU)
    t = gpu_ctx.fixedorsoln(alpha=0.4, sinc=0.3, solver=SOLVE_PLAIN, eps=1e-20, niter=1000)
    assert np.abs(r["amnp"] - t["amnp"]).max() <= 1e-7 * np.abs(t["amnp"]).max()


@pytest.mark.parametrize("n,x,spread", [(1, 0.05, 0.0), (17, 0.3, 0.0), (33, 0.9, 0.7), (100, 2.0, 0.0)])
def test_waits_that_run_out(n, x, spread):
    """No look at the other workgroups: every wait of the first panel runs out,
    and the factorization is done again without an exchange, on the context's
    first matrix.  Both routes take the same operations; their factors differ
    by rounding, times the condition (below 1e2) 1e-11."""
    from mstm_amd import geometry as G
    from mstm_amd.solver import SOLVE_LU, HipContext

    c = G.rsa_in_sphere(n, x, 0.15, seed=3, ri=1.31 + 0.01j)
    radius = c.radius.copy()
    radius[1::3] *= 1.0 - spread
    ctx = HipContext(0)
    try:
        ctx.set_spheres(c.pos, radius, c.ri, 1.0, 1e-6)
        ctx.set_lu_wait(0)
        r = ctx.fixedorsoln(alpha=0.4, sinc=0.3, solver=SOLVE_LU)
        ctx.set_lu_wait()
        ctx.clear()
        t = ctx.fixedorsoln(alpha=0.4, sinc=0.3, solver=SOLVE_LU)
        assert np.abs(r["amnp"] - t["amnp"]).max() <= 1e-11 * np.abs(t["amnp"]).max()
    finally:
        ctx.close()
