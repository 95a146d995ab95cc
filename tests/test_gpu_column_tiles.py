"""Column tiles whose exchange goes through LDS in two parts (the wide tiles), and
tiles whose lines are whole 128-byte cache lines, which are stored past the L2:
the same bits as the other tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIPE = 0x100  # MFX_COL_PIPELINED
ALT = 0x200  # MFX_COL_PLAN_ALT


# (line length, precision, widest plain tile, wide tile, radix plan): every wide tile
# there is; 17 columns leave a tile with a single column
@pytest.mark.parametrize("L,prec,plain,wide,plan",
                         [(288, "double", 8, 16, 0), (384, "double", 8, 16, 0), (512, "double", 8, 16, 0),
                          (768, "float", 8, 16, 0), (768, "double", 4, 8, 0), (1024, "double", 4, 8, 0),
                          (1536, "float", 4, 8, 0), (1536, "double", 2, 4, 0),
                          (384, "double", 8, 16, ALT), (768, "float", 8, 16, ALT), (768, "double", 4, 8, ALT),
                          (1024, "float", 8, 16, ALT), (1024, "double", 4, 8, ALT), (1536, "float", 4, 8, ALT),
                          (1536, "double", 2, 4, ALT)])
@pytest.mark.parametrize("flags", [0, PIPE])
def test_wide_tiles_equal_plain_ones(L, prec, plain, wide, plan, flags):
    import monofonic_amd as M
    print(f"wide tile L={L} {prec} flags {plan | flags:#x}", flush=True)
    ctx = M.Context(0)
    x = np.zeros((L, 3, 34))
    x[:, :, :32] = np.random.default_rng(L).standard_normal((L, 3, 32))
    out = []
    for w in (plain, wide):
        for inv in (0, 1):
            ctx.set_column_tile(L, prec, inv, w | plan | flags)
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


# M = 3n/2 lines at a pitch of whole cache lines.  A tile is streamed where its columns
# are whole lines too: 16 columns in FP32 and not 8, 8 in FP64 and not 4.  The set tile
# holds for every pass of the engine, the projections among them
@pytest.mark.parametrize("n,prec,cached,streamed", [(16, "float", 8, 16), (64, "float", 8, 16), (256, "double", 4, 8)])
@pytest.mark.parametrize("flags", [0, PIPE])
def test_streamed_lines_equal_cached_ones(orc, n, prec, cached, streamed, flags):
    import monofonic_amd as M
    from helpers import random_kspace_field
    print(f"streamed lines n={n} {prec} flags {flags:#x}", flush=True)
    phi_h = random_kspace_field(orc, n, 8, slope=-3.0)
    out = []
    for w in (cached, streamed):
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


# a field constant along y on (L, 16, 32) points, whose planes of 16 x 17 columns are
# whole cache lines, and on (L, 1, 32), whose planes are not: the sums over 16 equal
# values and the scales, powers of two apart, are exact
@pytest.mark.parametrize("L", [16, 96, 256, 512])
@pytest.mark.parametrize("prec,tile", [("float", 16), ("double", 8)])
@pytest.mark.parametrize("flags", [0, PIPE])
def test_streamed_planes_equal_cached_ones(L, prec, tile, flags):
    import monofonic_amd as M
    print(f"streamed planes L={L} {prec} flags {flags:#x}", flush=True)
    ctx = M.Context(0)
    for inv in (0, 1):
        ctx.set_column_tile(L, prec, inv, tile | flags)
    x = np.random.default_rng(L).standard_normal((L, 1, 32))
    k, r = [], []
    for n1 in (16, 1):
        a = np.zeros((L, n1, 34))
        a[:, :, :32] = x
        g = M.Grid_FFT(ctx, (L, n1, 32), (100.0, 100.0, 100.0), prec)
        g.upload(a)
        g.FourierTransformForward()
        k.append(g.kdata().copy())
        g.FourierTransformBackward()
        r.append(g.rdata().copy())
        del g
    assert np.array_equal(k[0][:, :1], 4 * k[1])
    assert not k[0][:, 1:].any()
    assert np.array_equal(r[0], np.broadcast_to(r[1], r[0].shape))
    ctx.close()
