"""Boundary flags and nearest-boundary distances through the hierarchy, at the
sizes where its passes can go wrong: rasters below, at and above a leaf (16
cells), a wave's strip (64 columns) and the levels a launch covers, long thin
rasters, no boundary at all, point counts around a wave, and points spread so
far that a wave's stack of nodes reaches its limit.  Flags against the
definition in numpy, distances against brute force: equal bit for bit."""
import numpy as np
import pytest

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu
NODATA = -9999.0


def flags_of(mask):
    v = np.zeros((mask.shape[0] + 2, mask.shape[1] + 2), bool)
    v[1:-1, 1:-1] = mask != NODATA
    inner = np.ones(mask.shape, bool)
    for dr in range(3):
        for dc in range(3):
            inner &= v[dr:dr + mask.shape[0], dc:dc + mask.shape[1]]
    return (v[1:-1, 1:-1] & ~inner).astype(np.uint8)


def brute(x, y, flags, xll, yll, cs):
    nr, nc = flags.shape
    xll, yll, cs = (np.float64(np.float32(v)) for v in (xll, yll, cs))
    cx = (xll + (np.arange(nc) + 0.5) * cs).astype(np.float32)
    cy = (yll + (np.float64(nr) - 0.5 - np.arange(nr)) * cs).astype(np.float32)
    r, c = np.nonzero(flags)
    if not len(r):
        return np.full(len(x), np.finfo(np.float64).max)
    out = np.empty(len(x))
    for k in range(len(x)):
        dx, dy = (cx[c] - x[k]).astype(np.float64), (cy[r] - y[k]).astype(np.float64)
        out[k] = (dx * dx + dy * dy).min()
    return out


def check(ctx, mask, n, seed, xll=0.0, yll=0.0, cs=1.0, spread=1.0):
    nr, nc = mask.shape
    rng = np.random.default_rng(seed)
    x = (xll + cs * nc * (0.5 + spread * rng.uniform(-0.6, 0.6, n))).astype(np.float32)
    y = (yll + cs * nr * (0.5 + spread * rng.uniform(-0.6, 0.6, n))).astype(np.float32)
    ctx.points_upload(x, y)
    ctx.mask_upload(M.grid(nc, nr, xll, yll, cs, NODATA), mask)
    want = flags_of(mask)
    d = ctx.CalcDist2Boundary()
    got, count = ctx.MarkBoundary()
    assert np.array_equal(got, want) and count == want.sum()
    assert np.array_equal(d, brute(x, y, want, xll, yll, cs))


@pytest.mark.parametrize("nr,nc", [(1, 1), (1, 16), (15, 17), (16, 16), (17, 15), (16, 64), (33, 65), (64, 63),
                                   (129, 257), (256, 256), (1, 3000), (2100, 3), (300, 511)])
def test_raster_sizes(ctx, nr, nc):
    rng = np.random.default_rng(nr * 10007 + nc)
    mask = np.where(rng.random((nr, nc)) < 0.9, np.float32(1.0), np.float32(NODATA))
    check(ctx, mask, 130, nr + nc, xll=3.25, yll=-7.5, cs=0.75)
    check(ctx, np.ones((nr, nc), np.float32), 70, nr + nc)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1000])
def test_point_counts(ctx, n):
    rr, cc = np.ogrid[0:200, 0:231]
    mask = np.where((rr - 99.5) ** 2 + (cc - 115) ** 2 < 80 ** 2, np.float32(1.0), np.float32(NODATA))
    check(ctx, mask, n, n)
    check(ctx, mask, n, n, spread=0.02)   # all near the centre: the whole circle is nearly equidistant


def test_no_boundary(ctx):
    check(ctx, np.full((40, 50), NODATA, np.float32), 66, 5)


def test_wide_waves_fill_the_stack(ctx):
    """64 points over a raster whose 17,000 leaves all hold boundary cells."""
    rng = np.random.default_rng(3)
    mask = np.where(rng.random((1900, 2300)) < 0.995, np.float32(1.0), np.float32(NODATA))
    check(ctx, mask, 64, 11)
    check(ctx, mask, 200, 12)


def test_coarse_coordinates(ctx):
    """Far from the origin many cell centres round to the same float."""
    rng = np.random.default_rng(4)
    mask = np.where(rng.random((90, 110)) < 0.8, np.float32(1.0), np.float32(NODATA))
    check(ctx, mask, 200, 13, xll=1.0e6, yll=-2.0e6, cs=0.03)
