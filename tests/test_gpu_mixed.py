"""The mixed-radix kernels (fft_mixed.hpp) at the lengths and row counts where
their schedules change: two to four stages, each radix, an odd number of rows
(a pair with one row), tiles with fewer columns than their width, the longest
lines."""
import numpy as np
import pytest

from conftest import rel_max, rel_rms

pytestmark = pytest.mark.gpu


# a transform of length L errs by about eps log2(L) in the rms: 1e-13 is 40
# times that of FP64 at L = 2000, 3e-6 four times that of FP32
@pytest.mark.parametrize("shape", [(4, 6, 10), (9, 5, 14), (7, 21, 50), (25, 3, 42), (20, 28, 70), (45, 49, 126),
                                   (625, 3, 18), (2000, 2, 60), (3, 1200, 30), (5, 3, 2000), (150, 162, 250)])
@pytest.mark.parametrize("prec,tol", [("double", 1e-13), ("float", 3e-6)])
def test_transforms_vs_numpy(ctx, shape, prec, tol):
    import monofonic_amd as M
    n0, n1, n2 = shape
    print(f"mixed r2c/c2r {shape} {prec}", flush=True)
    rng = np.random.default_rng(n0 + 7 * n1 + 13 * n2)
    x = rng.standard_normal(shape)
    a = np.zeros((n0, n1, n2 + 2))
    a[:, :, :n2] = x
    g = M.Grid_FFT(ctx, shape, (100.0, 100.0, 100.0), prec)
    g.upload(a)
    g.FourierTransformForward()
    ref = np.fft.rfftn(x) / np.sqrt(n0 * n1 * n2)
    got = g.kdata()
    assert rel_rms(got, ref) < tol and rel_max(got, ref) < 20 * tol
    g.FourierTransformBackward()
    back = g.download()
    assert rel_max(back[:, :, :n2], x) < 20 * tol
    assert np.all(back[:, :, n2:] == 0)
