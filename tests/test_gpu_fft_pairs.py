"""Near-field pair translations of the FFT product, one kernel per order: three
spheres whose cells are all neighbours, so the FFT product is the sum over the
pairs and equals the direct product up to the rounding of the FP32 spectrum
(the periodic grid's other offsets), for which test_gpu_fft.py allows 1e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,x,eps", [(1, 0.05, 1e-1), (2, 0.05, 1e-4), (3, 0.3, 1e-5), (4, 1.0, 1e-6),
                                         (5, 2.0, 1e-6), (6, 2.0, 1e-7), (7, 3.0, 1e-7), (8, 4.0, 1e-7)])
def test_pairs_match_direct(gpu_ctx, order, x, eps):
    from mstm_amd.solver import FP32, FP64

    pos = np.array([[0.0, 0.0, 0.0], [2.2, 0.1, 0.2], [1.0, 2.1, -0.3]]) * x
    gpu_ctx.set_spheres(pos, np.array([1.0, 0.9, 0.5]) * x, np.full(3, 1.5 + 0.01j), 1.0, eps)
    assert max(gpu_ctx.orders()[0]) == order
    gpu_ctx.node_selection(0.0, -1, 2)
    ne = gpu_ctx.number_eqns
    rng = np.random.default_rng(order)
    a = rng.normal(size=(2, ne)) + 1j * rng.normal(size=(2, ne))
    args = (a, [False, True], [True, True])
    d = gpu_ctx.sphereinteraction(*args, precision=FP64)
    for prec in (FP64, FP32):
        gpu_ctx.setup_fft(prec)
        f = gpu_ctx.sphereinteraction(*args, fft_option=True, precision=prec)
        assert np.abs(f - d).max() <= 1e-5 * np.abs(d).max()
