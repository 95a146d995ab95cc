"""Column tiles whose exchange goes through LDS in two parts (the wide tiles), and
tiles whose lines are whole 128-byte cache lines, which are stored past the L2:
the same bits as the other tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIPE = 0x100  # MFX_COL_PIPELINED
ALT = 0x200  # MFX_COL_PLAN_ALT


# (line length, precision, widest plain tile, wide tile): the lengths whose wide
# tile exists; 17 columns leave a tile with a single column
@pytest.mark.parametrize("L,prec,plain,wide", [(512, "double", 8, 16), (768, "float", 8, 16), (768, "double", 4, 8),
                                               (1024, "float", 8, 16), (1536, "float", 4, 8), (1536, "double", 2, 4)])
@pytest.mark.parametrize("flags", [0, PIPE])
def test_wide_tiles_equal_plain_ones(L, prec, plain, wide, flags):
    import monofonic_amd as M
    print(f"wide tile L={L} {prec} flags {flags:#x}", flush=True)
    ctx = M.Context(0)
    x = np.zeros((L, 3, 34))
    x[:, :, :32] = np.random.default_rng(L).standard_normal((L, 3, 32))
    out = []
    for w in (plain, wide):
        for inv in (0, 1):
            try:
                ctx.set_column_tile(L, prec, inv, w | flags)
            except M.MfxError:
                pytest.skip("no such tile at this length")
        g = M.Grid_FFT(ctx, (L, 3, 32), (100.0, 100.0, 100.0), prec)
        g.upload(x)
        g.FourierTransformForward()
        k = g.download().copy()
        g.FourierTransformBackward()
        out.append((k, g.download().copy()))
        del g
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
    ctx.close()


# M = 3n/2 lines at a pitch of whole cache lines: 4 columns are always part of one,
# 8 are one in FP64 only, 16 in both
@pytest.mark.parametrize("n,prec", [(16, "float"), (16, "double"), (64, "float"), (64, "double"), (96, "double")])
@pytest.mark.parametrize("flags", [0, PIPE])
def test_streamed_lines_equal_cached_ones(orc, n, prec, flags):
    import monofonic_amd as M
    from helpers import random_kspace_field
    print(f"streamed lines n={n} {prec} flags {flags:#x}", flush=True)
    phi_h = random_kspace_field(orc, n, 8, slope=-3.0)
    out = []
    for w in (8, 16):
        ctx = M.Context(0)
        for inv in (0, 1):
            ctx.set_column_tile(3 * n // 2, prec, inv, w | flags)
        grids = [M.Grid_FFT(ctx, n, 100.0, prec, initialspace=M.kspace_id) for _ in range(6)]
        grids[0].upload(phi_h)
        conv = M.OrszagConvolver(ctx, n, 100.0, prec)
        conv.lpt_sources(grids[0], grids[1], grids[2], grids[3:], 3)
        out.append([g.kdata().copy() for g in grids[1:]])
        del conv, grids
        ctx.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
