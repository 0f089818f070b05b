"""T-matrix columns solved in blocks (plain solver) against the pair-by-pair
mixed solver: one sphere, one and several sphere blocks with remainders,
spheres of unequal order, and a cluster whose degrees take several blocks of
unequal width.

Both stop at |r|^2/|b|^2 < 1e-14, so each column carries a relative residual of
1e-7 at most; times a condition below 1e2 that is 1e-5 of the largest element."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cluster(n, x, spread):
    from mstm_amd import geometry as G

    c = G.rsa_in_sphere(n, x, 0.12, seed=11, ri=1.5 + 0.01j)
    radius = c.radius.copy()
    radius[1::3] *= 1.0 - spread
    return c.pos, radius, c.ri


@pytest.mark.parametrize("n,x,spread", [(1, 1.0, 0.0), (2, 0.3, 0.0), (16, 0.8, 0.5), (17, 1.2, 0.0), (40, 0.6, 0.3),
                                        (300, 2.2, 0.2)])
def test_blocks_match_pairs(gpu_ctx, n, x, spread):
    from mstm_amd.solver import SOLVE_MIXED, SOLVE_PLAIN

    gpu_ctx.set_spheres(*_cluster(n, x, spread), 1.0, 1e-6)
    r = gpu_ctx.tmatrix_solution(eps=1e-14, niter=2000, conveps=1e-3, solver=SOLVE_PLAIN)
    m = gpu_ctx.tmatrix_solution(eps=1e-14, niter=2000, conveps=1e-3, solver=SOLVE_MIXED)
    assert r["istat"] == 0 and r["T"] == m["T"]
    for k in ("tmat", "sqeff", "qteff"):
        assert np.abs(r[k] - m[k]).max() <= 1e-5 * np.abs(m[k]).max(), k


def test_blocks_iteration_limit(gpu_ctx):
    gpu_ctx.set_spheres(*_cluster(40, 1.0, 0.0), 1.0, 1e-6)
    r = gpu_ctx.tmatrix_solution(eps=1e-14, niter=3, conveps=1e-3)
    assert r["istat"] == 1 and r["maxiter"] == 4 and r["maxerr"] > 1e-14


def test_blocks_are_in_the_statistics(gpu_ctx):
    """Tile times and products of the blocks, above the 500 spheres up to which
    single systems are replayed from graphs: one start per column pair, one
    four-column product per iteration of a pair."""
    gpu_ctx.set_spheres(*_cluster(520, 0.2, 0.0), 1.0, 1e-3)
    gpu_ctx.clear()
    r = gpu_ctx.tmatrix_solution(eps=1e-6, conveps=1e-3)
    st = gpu_ctx.stats()
    assert st["tile_launches_fp64"] > 0 and st["tile4_launches_fp64"] > 0
    assert 0.0 < st["tile_ms_fp64"] + st["tile4_ms_fp64"] < st["tmatrix_ms"]
    pairs = st["tmatrix_solves"] // 2
    assert pairs == sum(2 * l + 1 for l in range(1, r["T"] + 1))
    assert pairs + st["iters_fp64"] / 2 <= st["matvecs_fp64"] <= pairs + st["iters_fp64"]


def test_blocks_give_their_work_space_back():
    """The block work space (300 MB here) goes with the spheres it was for, so
    that the next cluster has the room; what stays is a single pair's."""
    import ctypes as C

    from mstm_amd.solver import HipContext

    ctx = HipContext(0)

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert C.CDLL(ctx.L._name).hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    try:
        one = (np.zeros((1, 3)), np.ones(1), np.full(1, 1.5 + 0.01j), 1.0, 1e-6)
        ctx.set_spheres(*one)
        free0 = free()
        ctx.set_spheres(*_cluster(200, 0.6, 0.0), 1.0, 1e-6)
        ctx.tmatrix_solution(conveps=1e-3)
        held = free0 - free()
        ctx.set_spheres(*one)
        left = free0 - free()
        print(f"held {held >> 20} MB with the T-matrix, {left >> 20} MB after")
        assert left < (128 << 20)
    finally:
        ctx.close()
