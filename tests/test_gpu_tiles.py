"""GPU products of the direct tiles at every compiled sphere order, against the
C oracle: one to four columns, clusters below, at and above whole blocks of 16
spheres (padded blocks, diagonal tiles only, step groups), mixed orders.

Tolerances, by the precision of the form (max-norm relative): FP64 1e-10,
FP32 2e-5, as for the other products."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# size parameter -> order 1..8 at m = 1.4+0.01i and mie_epsilon eps
CASES = [(0.02, 1e-2, 1), (0.3, 1e-4, 2), (0.4, 1e-6, 3), (1.2, 1e-6, 4), (2.0, 1e-6, 5), (2.8, 1e-6, 6),
         (3.6, 1e-6, 7), (4.6, 1e-6, 8)]


@pytest.mark.parametrize("n", [1, 16, 17, 50])
@pytest.mark.parametrize("x,eps,order", CASES)
def test_tile_products_match_oracle(gpu_ctx, x, eps, order, n):
    from mstm_amd import geometry as G
    from mstm_amd.solver import FP32, FP64, FP64_FP32
    from oracle.oracle import OracleCluster

    c = G.rsa_in_sphere(n, x, 0.2, seed=90 + n, ri=1.4 + 0.01j) if n > 1 else G.Cluster(
        np.zeros((1, 3)), np.full(1, x), np.full(1, 1.4 + 0.01j))
    rad = c.radius.copy()
    rad[1::3] *= 0.7  # a third of the spheres of lower order
    o, _ = gpu_ctx.set_spheres(c.pos, rad, c.ri, 1.0, eps)
    assert o.max() == order, o.max()
    oc = OracleCluster(c.pos, rad, c.ri, 1.0, eps)
    gpu_ctx.setup_direct(FP64_FP32)
    rng = np.random.default_rng(order)
    a = rng.normal(size=(5, gpu_ctx.number_eqns)) + 1j * rng.normal(size=(5, gpu_ctx.number_eqns))
    ct, mm = [False, True, True, False, True], [True, True, False, False, True]
    ref = oc.sphereinteraction(a, ct, mm)
    for prec, tol in ((FP64, 1e-10), (FP32, 2e-5)):
        for ncol in (1, 2, 3, 5):
            out = gpu_ctx.sphereinteraction(a[:ncol], ct[:ncol], mm[:ncol], precision=prec)
            if n == 1:
                assert not out.any()
                continue
            for r in range(ncol):
                assert np.abs(out[r] - ref[r]).max() <= tol * np.abs(ref[r]).max(), (prec, ncol, r)
