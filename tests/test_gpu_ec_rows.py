"""Edge-correction weights where a row's chord meets cell centres: cell sizes
that are and are not powers of two, points exactly on centres and edges,
bandwidths whose cut-off falls on centres (3h a whole number of cells), boxes
below, at and above a column chunk, rows with no, one and several runs, points
outside the raster, and origins so far away that centres are coarse.  The
number of cells inside is exact; the weight against 64 bits.  Cells are taken
from the estimator's own box of 3h around a point, whose corners truncate."""
import numpy as np
import pytest

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu
NODATA = -9999.0
TWO_PI_F = np.float64(np.float32(6.2831853071795862))
# half an ulp of the weight, and per cell the rounding of two exponent arguments
# (6.5 in base 2 each: 4.5 2^-24 relative) and two exponentials (2^-23 each)
RTOL = (1 + 2 * 4.5 + 4) * 2.0 ** -24


def want(x, y, h, mask, xll, yll, cs):
    nr, nc = mask.shape
    xll, yll, cs = (np.float64(np.float32(v)) for v in (xll, yll, cs))
    cx = (xll + (np.arange(nc) + 0.5) * cs).astype(np.float32)
    cy = (yll + (np.float64(nr) - 0.5 - np.arange(nr)) * cs).astype(np.float32)
    valid = mask != NODATA
    ew, count = np.empty(len(x)), 0
    for i in range(len(x)):
        # the box, with its unsigned upper ends
        px, py, r3 = np.float64(x[i]), np.float64(y[i]), 3.0 * np.float64(h[i])
        top, bot = int((py + r3 - yll) / cs), int((py - r3 - yll) / cs)
        left, right = int((px - r3 - xll) / cs), int((px + r3 - xll) / cs)
        rows, cols = np.arange(nr), np.arange(nc)
        box = ((rows >= nr - 1 - top) & ((rows <= nr - 1 - bot) | (bot > nr - 1)))[:, None] \
            & ((cols >= left) & ((cols <= right) | (right < 0)))[None, :]
        h2 = np.float64(h[i] * h[i])
        dx = (cx - x[i]).astype(np.float64) ** 2
        dy = (cy - y[i]).astype(np.float64) ** 2
        ins = box & valid & (dx[None, :] + dy[:, None] < 9.0 * h2)
        k = np.exp(dy / (-2 * h2))[:, None] * np.exp(dx / (-2 * h2))[None, :]
        with np.errstate(divide="ignore"):
            ew[i] = 1.0 / (k[ins].sum() * np.float64(np.float32(cs) * np.float32(cs)) / (h2 * TWO_PI_F))
        count += int(ins.sum())
    return ew, count


def check(ctx, x, y, h, mask, xll=0.0, yll=0.0, cs=1.0):
    nr, nc = mask.shape
    ctx.points_upload(x, y)
    ctx.mask_upload(M.grid(nc, nr, xll, yll, cs, NODATA), mask)
    ctx.set_dist_to_boundary(np.zeros(len(x)))   # every point is corrected
    ctx.set_bandwidths(h)
    got, n_eval = ctx.EdgeCorrectionWeightsExact()
    ref, count = want(x, y, h, mask, xll, yll, cs)
    assert n_eval == count
    inside = np.isfinite(ref)
    assert np.all(np.isinf(got[~inside]))
    assert np.all(np.abs(got[inside] - ref[inside]) <= RTOL * ref[inside])


def holed(nr, nc, seed):
    r = np.random.default_rng(seed)
    m = np.ones((nr, nc), np.float32)
    for _ in range(12):
        a, b = r.integers(0, nr), r.integers(0, nc)
        m[a:a + 9, b:b + 7] = NODATA
    m[nr // 2] = NODATA
    return m


@pytest.mark.parametrize("cs", [1.0, 0.25, 2.5, 0.3])
def test_cell_sizes(ctx, cs):
    r = np.random.default_rng(int(cs * 100))
    n = 120
    x, y = (r.uniform(-20 * cs, 180 * cs, n).astype(np.float32) for _ in range(2))
    h = (cs * np.exp(r.uniform(-1.0, 3.5, n))).astype(np.float32)
    check(ctx, x, y, h, holed(130, 170, 1), 0.0, 0.0, cs)


def test_chords_ending_on_centres(ctx):
    """Points on centres, edges and corners, cut-off radii of whole cells."""
    k = np.arange(12)
    x = np.concatenate([20.5 + k, 20.0 + k, 20.25 + k]).astype(np.float32)
    y = np.concatenate([30.5 + k, 30.0 + k, 30.5 + 0 * k]).astype(np.float32)
    for radius in (1.0, 5.0, 13.0, 25.0):
        h = np.full(36, radius, np.float32) / np.float32(3.0)
        check(ctx, x, y, h, np.ones((64, 64), np.float32))
        check(ctx, x, y, h, holed(64, 64, 5))


@pytest.mark.parametrize("nc", [1023, 1024, 1025, 1100, 2300])
def test_box_widths_around_a_chunk(ctx, nc):
    r = np.random.default_rng(nc)
    x = np.array([0.0, nc / 2, nc - 0.5, nc / 3], np.float32)
    y = r.uniform(0, 40, 4).astype(np.float32)
    for h in (170.4, 170.7, 341.2, 900.0):
        check(ctx, x, y, np.full(4, h, np.float32), holed(41, nc, nc))


@pytest.mark.parametrize("xll,cs", [(4.0e5, 0.05), (1.0e6, 0.02), (-3.0e6, 30.0)])
def test_far_origins(ctx, xll, cs):
    r = np.random.default_rng(9)
    x = (xll + cs * r.uniform(0, 100, 60)).astype(np.float32)
    y = (cs * r.uniform(0, 80, 60)).astype(np.float32)
    h = (cs * np.exp(r.uniform(0.0, 3.0, 60))).astype(np.float32)
    check(ctx, x, y, h, holed(80, 100, 3), xll, 0.0, cs)
