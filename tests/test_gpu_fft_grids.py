"""FFT product on grids at the edges of its transforms: one-point axes, odd and
5-smooth lengths, an xy plane or a z axis too long for the fused kernels in FP64
only (24x24, 120) or in both precisions (36x36, 240).

Both precisions against the C oracle, which sums over the grid's nodes without
any transform.  The products share an FP32 spectrum (relative rounding 6e-8)
and sum a few hundred terms: 1e-5 of the largest element, as in
test_gpu_fft.py; a misplaced element is of order one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,fva,cells", [((12, 12, 1), 0.0, (24, 24, 1)), ((24, 24, 1), 0.1, (36, 36, 1)),
                                            ((1, 1, 80), 0.1, (1, 1, 120)), ((1, 1, 80), 0.0, (1, 1, 240)),
                                            ((9, 7, 5), 0.0, (10, 8, 5)), ((9, 7, 5), 0.1, (15, 10, 8)),
                                            ((30, 3, 3), 0.1, (45, 4, 4)), ((3, 30, 2), 0.0, (3, 45, 2))])
def test_fft_product(gpu_ctx, dims, fva, cells):
    from mstm_amd.solver import FP32, FP64
    from oracle.oracle import OracleCluster

    rng = np.random.default_rng(1)
    g = np.stack(np.meshgrid(*[np.arange(d) for d in dims], indexing="ij"), -1).reshape(-1, 3) * 2.6
    pos = g + rng.uniform(-0.15, 0.15, g.shape)
    n = len(pos)
    gpu_ctx.set_spheres(pos, np.full(n, 0.5), np.full(n, 1.5 + 0.01j), 1.0, 1e-6)
    assert tuple(gpu_ctx.node_selection(fva, -1, 2)["cell_dim"]) == cells
    ne = gpu_ctx.number_eqns
    a = rng.normal(size=(2, ne)) + 1j * rng.normal(size=(2, ne))
    args = (a, [False, True], [True, True])
    oc = OracleCluster(pos, np.full(n, 0.5), np.full(n, 1.5 + 0.01j), 1.0, 1e-6)
    assert tuple(oc.node_selection(fva, -1, 2)["cell_dim"]) == cells
    ref = oc.sphereinteraction(*args, use_fft=True)
    out = {}
    for prec in (FP64, FP32):
        gpu_ctx.setup_fft(prec)
        out[prec] = gpu_ctx.sphereinteraction(*args, fft_option=True, precision=prec)
        for r in range(2):
            assert np.abs(out[prec][r] - ref[r]).max() <= 1e-5 * np.abs(ref[r]).max(), (prec, r)
    assert np.abs(out[FP64] - out[FP32]).max() <= 1e-5 * np.abs(out[FP64]).max()
