"""Passes over several arrays in one launch: the particle components and the 3a
intermediates and sources of the LPT engine, at the grid sizes where the arrays
taken together change (six, three, two and one; four, two and one), and the x
passes whose columns are a whole plane."""
import numpy as np
import pytest

from conftest import rel_rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,prec", [(16, "float"), (64, "double"), (160, "float"), (160, "double"), (192, "float"),
                                    (192, "double"), (224, "double"), (44, "float")])
def test_particle_components_equal_one_at_a_time(ctx, n, prec):
    """with baryons every component is transformed on its own, from the same
    assembled values and by the same kernels: the same bits"""
    import monofonic_amd as M
    print(f"components n={n} {prec}", flush=True)
    kw = dict(LPTorder=2, precision=prec, generator="NGENIC", seed=3)
    ics = [M.ICGenerator(ctx, n, 2.0 * n, 24.0, DoBaryons=b, **kw) for b in (False, True)]
    for ic in ics:
        ic.run()
    for w in range(6):
        assert np.array_equal(ics[0].particles(w), ics[1].particles(w)), w


@pytest.mark.parametrize("n,prec,path", [(32, "double", "stored"), (96, "double", "stored"), (128, "double", "stored"),
                                         (128, "double", "streamed"), (192, "double", "stored"),
                                         (192, "double", "streamed"), (160, "double", "stored")])
def test_lpt_groups_vs_sequence(ctx, orc, n, prec, path):
    """the engine against the reference's call sequence through the named
    convolutions: regrouped sums of the same products, 1e-12 in the rms"""
    import monofonic_amd as M
    from helpers import random_kspace_field
    from test_gpu_lpt import gpu_lpt_reference_sequence
    print(f"lpt groups n={n} {prec} {path}", flush=True)
    phi = M.Grid_FFT(ctx, n, 100.0, prec, initialspace=M.kspace_id)
    phi.upload(random_kspace_field(orc, n, 31, slope=-3.0))
    conv = M.OrszagConvolver(ctx, n, 100.0, prec)
    conv.set_lpt_path(path)
    sets = [[M.Grid_FFT(ctx, n, 100.0, prec, initialspace=M.kspace_id) for _ in range(5)] for _ in range(2)]
    conv.lpt_sources(phi, sets[0][0], sets[0][1], tuple(sets[0][2:]), order=3)
    gpu_lpt_reference_sequence(M, conv, phi, sets[1][0], sets[1][1], sets[1][2:], 3)
    for a, b in zip(*sets):
        assert rel_rms(a.kdata(), b.kdata()) < 1e-12


@pytest.mark.parametrize("shape", [(16, 3, 6), (24, 5, 2), (32, 1, 32), (64, 7, 30), (96, 33, 18), (512, 2, 4),
                                   (1536, 3, 2)])
@pytest.mark.parametrize("prec,tol", [("double", 1e-13), ("float", 3e-6)])
def test_plane_columns_vs_numpy(ctx, shape, prec, tol):
    """planes that are no multiple of a tile, and smaller than one"""
    import monofonic_amd as M
    n0, n1, n2 = shape
    print(f"plane columns {shape} {prec}", flush=True)
    x = np.random.default_rng(n0 + n1 + n2).standard_normal(shape)
    a = np.zeros((n0, n1, n2 + 2))
    a[:, :, :n2] = x
    g = M.Grid_FFT(ctx, shape, (100.0, 100.0, 100.0), prec)
    g.upload(a)
    g.FourierTransformForward()
    assert rel_rms(g.kdata(), np.fft.rfftn(x) / np.sqrt(x.size)) < tol
    g.FourierTransformBackward()
    assert rel_rms(g.rdata(), x) < 2 * tol
