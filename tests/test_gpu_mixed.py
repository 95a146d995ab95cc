"""The mixed-radix kernels (fft_mixed.hpp) at the lengths and row counts where
their schedules change: two to four stages, each radix, an odd number of rows
(a pair with one row), tiles with fewer columns than their width, the longest
lines; and the fused LPT engine on the padded lengths that run them."""
import numpy as np
import pytest

from conftest import rel_max, rel_rms
from helpers import random_kspace_field

pytestmark = pytest.mark.gpu

BOX = 100.0


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


def _fields(M, ctx, orc, n, prec):
    phi_h = random_kspace_field(orc, n, n, slope=-3.0)
    phi = M.Grid_FFT(ctx, n, BOX, prec, initialspace=M.kspace_id)
    phi.upload(phi_h)
    out = [M.Grid_FFT(ctx, n, BOX, prec, initialspace=M.kspace_id) for _ in range(5)]
    return phi_h, phi, out


# padded lengths 30, 42, 54, 60, 90, 150, 180: schedules of one to three stages
# before the fixed last radix (6 in FP32, 3 in FP64)
@pytest.mark.parametrize("n", [20, 28, 36, 40, 60, 100, 120])
@pytest.mark.parametrize("prec,rms,mx", [("double", 1e-12, 1e-10), ("float", 2e-5, 2e-3)])
@pytest.mark.parametrize("order", [2, 3])
def test_lpt_engine_vs_oracle(ctx, orc, n, prec, rms, mx, order):
    import monofonic_amd as M
    print(f"mixed lpt engine n={n} {prec} order={order}", flush=True)
    phi_h, phi, (phi2, phi3, *A3) = _fields(M, ctx, orc, n, prec)
    conv = M.OrszagConvolver(ctx, n, BOX, prec)
    if order == 2:
        conv.lpt_sources(phi, phi2, order=2)
    else:
        conv.lpt_sources(phi, phi2, phi3, tuple(A3), order=3)
        assert conv.lpt_path == "stored"  # the engine ran, not the convolve sequence
    r2, r3, rA = orc.lpt_terms(phi_h, BOX, order)
    pairs = [(phi2, r2)] + ([(phi3, r3)] + list(zip(A3, rA)) if order == 3 else [])
    for got, ref in pairs:
        assert rel_rms(got.kdata(), orc.kview(ref)) < rms
        assert rel_max(got.kdata(), orc.kview(ref)) < mx


@pytest.mark.parametrize("n", [20, 28, 60, 100])
def test_lpt_streamed_request_keeps_the_sequence(ctx, orc, n):
    """the mixed-radix stages have no streamed 3LPT path: asked for it, such a
    size runs the convolve sequence, which the engine agrees with"""
    import monofonic_amd as M
    phi_h, phi, (phi2, phi3, *A3) = _fields(M, ctx, orc, n, "double")
    conv = M.OrszagConvolver(ctx, n, BOX, "double")
    conv.set_lpt_path("streamed")
    conv.lpt_sources(phi, phi2, phi3, tuple(A3), order=3)
    seq = [g.kdata().copy() for g in (phi2, phi3, *A3)]
    conv.set_lpt_path("stored")
    conv.lpt_sources(phi, phi2, phi3, tuple(A3), order=3)
    for g, s in zip((phi2, phi3, *A3), seq):
        assert rel_rms(g.kdata(), s) < 1e-12


@pytest.mark.parametrize("shape", [(20, 16, 40), (150, 16, 32), (35, 20, 16), (70, 16, 300)])
@pytest.mark.parametrize("prec", ["float", "double"])
def test_constant_field_has_one_mode(ctx, shape, prec):
    """the butterflies cancel a line's mean exactly, with rounded constants too
    (lengths of two and more mixed-radix stages; single primes run other kernels)"""
    import monofonic_amd as M
    print(f"constant field {shape} {prec}", flush=True)
    a = np.zeros(shape[:2] + (shape[2] + 2,))
    a[:, :, :shape[2]] = 1.0
    g = M.Grid_FFT(ctx, shape, (100.0, 100.0, 100.0), prec)
    g.upload(a)
    g.FourierTransformForward()
    k = g.kdata().copy()
    assert abs(k[0, 0, 0] / np.sqrt(np.prod(shape)) - 1) < 1e-6
    k[0, 0, 0] = 0
    assert not k.any()


# A line of mean 1 with 1 % fluctuations: its longest waves are formed from
# differences, so that they err by what rounds at the size of the fluctuations.  In
# units of 2^-24 (2^-53) of the transform of those, a restatement in single
# precision gives an rms of 1.3 to 1.7 for schedules that start with 8 or 4 and up
# to 2.3 for the ones of these lengths; where the first radix adds raw values and
# subtracts the sums it is 30 to 45.
@pytest.mark.parametrize("L", [120, 126, 162, 225, 240, 300, 360, 375, 567])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("prec,bits", [("double", 53), ("float", 24)])
def test_mean_stays_out_of_the_longest_waves(ctx, L, axis, prec, bits):
    import monofonic_amd as M
    if axis == 2 and L % 2:
        pytest.skip("rows are even")
    print(f"mean and fluctuations L={L} axis {axis} {prec}", flush=True)
    # x lines: one line, constant along y and z, so that the passes before are exact;
    # y lines: four; z rows: sixteen
    shape = [(L, 4, 4), (4, L, 4), (4, 4, L)][axis]
    lines = [(L, 1, 1), (4, L, 1), (4, 4, L)][axis]
    w = np.exp(-2j * np.arange(L, dtype=np.longdouble) * (4 * np.arctan(np.longdouble(1))) / L)
    sums = []
    for seed in range((48, 16, 8)[axis]):
        x = 1 + 0.01 * np.random.default_rng(100 * L + seed).standard_normal(lines)
        x = x.astype(np.float32 if prec == "float" else np.float64)
        a = np.zeros(shape[:2] + (shape[2] + 2,))
        a[:, :, :shape[2]] = x
        g = M.Grid_FFT(ctx, shape, (100.0, 100.0, 100.0), prec)
        g.upload(a)
        g.FourierTransformForward()
        k = g.kdata() * np.sqrt(np.prod(shape))
        one = np.tensordot(x.astype(np.longdouble), w, axes=([axis], [0]))
        if axis == 0:
            got, ref = np.array([k[1, 0, 0], k[-1, 0, 0]]), 16 * np.array([one[0, 0], np.conj(one[0, 0])])
        elif axis == 1:
            ref = np.array([np.fft.fft(one[:, 0].astype(complex)), np.fft.fft(np.conj(one[:, 0]).astype(complex))])
            got, ref = np.array([k[:, 1, 0], k[:, -1, 0]]), 4 * ref
        else:
            got, ref = k[:, :, 1], np.fft.fft2(one.astype(complex))
        # of one line's transform: the other axes' modes are sums over their lines
        e = np.abs(got - ref.astype(complex)) / (16, 8, 4)[axis]
        sums.append(np.mean(e ** 2))
    unit = 2.0 ** -bits * 0.01 * np.sqrt(L)
    assert np.sqrt(np.mean(sums)) / unit < 4


def source_by_products(M, ctx, k, n, prec):
    """the 2LPT source through the named convolutions, one product after another"""
    a = np.zeros((n, n, n + 2))
    a.view(np.complex128)[...] = k
    phi, out = (M.Grid_FFT(ctx, n, BOX, prec, initialspace=M.kspace_id) for _ in range(2))
    phi.upload(a)
    conv, op = M.OrszagConvolver(ctx, n, BOX, prec), M.op
    conv.convolve_SumOfHessians(phi, (0, 0), phi, (1, 1), (2, 2), op.assign_to(out))
    conv.convolve_Hessians(phi, (1, 1), phi, (2, 2), op.add_to(out))
    for d in ((0, 1), (0, 2), (1, 2)):
        conv.convolve_Hessians(phi, d, phi, d, op.subtract_from(out))
    return out.kdata().copy()


def long_wave_errors(M, ctx, n, seeds):
    """rms over `seeds` realisations of the FP32 second-order potential's error
    against FP64, by shells q = 1, 2, 3 of (2 pi / L)^2 q, relative to the field"""
    i = np.fft.fftfreq(n) * n
    q = i[:, None, None] ** 2 + i[None, :, None] ** 2 + np.arange(n // 2 + 1)[None, None, :] ** 2
    q[0, 0, 0] = 1
    err = np.zeros(3)
    for seed in range(seeds):
        k = np.fft.rfftn(np.random.default_rng(seed).standard_normal((n, n, n))) / np.sqrt(n ** 3) / q ** 1.5
        k[0, 0, 0] = 0
        k = k.astype(np.complex64).astype(np.complex128)
        f, d = (source_by_products(M, ctx, k, n, prec) / q for prec in ("float", "double"))
        f[0, 0, 0] = d[0, 0, 0] = 0
        e = np.abs(f - d) ** 2 / np.sum(np.abs(d) ** 2)
        for s in range(3):
            err[s] += np.sum(e[(q > s + 0.5) & (q < s + 1.5)]) / seeds
    return np.sqrt(err)


# the direct-DFT kernels that ran these sizes before erred by so much over the same
# seeds; the second and third shell hold more modes but vary by a fifth between sets of
# seeds
@pytest.mark.parametrize("n,seeds,before", [(40, 24, (1.66e-7, 8.2e-8, 4.0e-8)), (100, 12, (2.87e-7, 1.35e-7, 7.7e-8)),
                                            (160, 8, (2.83e-7, 8.9e-8, 4.6e-8))])
def test_long_waves_of_convolutions(ctx, n, seeds, before):
    import monofonic_amd as M
    print(f"long waves of products n={n}", flush=True)
    err = long_wave_errors(M, ctx, n, seeds)
    assert err[0] < before[0]
    assert np.all(err[1:] < 1.25 * np.array(before[1:]))
