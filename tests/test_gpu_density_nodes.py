"""Density rasters whose wide kernels are summed at nodes of each block: large
candidate lists (cut and uncut blocks, ragged edges, a single column or row in the
last block), bandwidths on both sides of the smallest that goes to the nodes,
cell sizes, masks, tiles.  Against the sum in 64 bits with the exact cut-off at
cells of every block."""
import numpy as np
import pytest

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu
TWO_PI_F = np.float64(np.float32(6.2831853071795862))

# error of a cell or node sum, relative to it: 2^-24 for the rounding of the
# result, of a coefficient and of each factor's argument (times at most 4.5, in
# base 2 6.5), two of each exponential, the product, 64 terms of a float sum
RTOL = (1 + 1 + 6.5 + 6.5 + 2 + 2 + 1 + 64) * 2.0 ** -24
# a cell takes the 16 x 16 nodes with weights whose sizes add up to 2.73 per
# dimension; 4.4e-9 for the interpolation
AMP = 2.73 ** 2


def want(x, y, coef, h2, cx, cy):
    out = np.zeros(len(cx))
    for i in range(0, len(cx), 64):
        dx = (cx[i:i + 64, None] - x[None, :]).astype(np.float64)
        dy = (cy[i:i + 64, None] - y[None, :]).astype(np.float64)
        d2 = dx * dx + dy * dy
        out[i:i + 64] = np.where(d2 < 9.0 * h2, np.exp(d2 / (-2.0 * h2)) * coef, 0.0).sum(1)
    return out


def check(ctx, n, ncols, nrows, cs, h_lo, h_hi, mask=False, tile=None, seed=1):
    r = np.random.default_rng(seed)
    x = r.uniform(0, ncols * cs, n).astype(np.float32)
    y = r.uniform(0, nrows * cs, n).astype(np.float32)
    w = r.uniform(0.5, 2.0, n).astype(np.float32)
    hs = np.exp(r.uniform(np.log(h_lo * cs), np.log(h_hi * cs), n)).astype(np.float32)
    ctx.points_upload(x, y, w)
    ctx.set_bandwidths(hs)
    ctx.set_ec_weights(None)
    m = None
    if mask:
        m = np.ones((nrows, ncols), np.float32)
        m[r.random((nrows, ncols)) < 0.1] = -9999.0
    if tile:
        gt = [0.0, cs, 0.0, nrows * cs, 0.0, -cs]
        den = ctx.KernelDensityEstimation_raster(ncols, nrows, gt, -9999.0, tile, tile, m)
    else:
        den = ctx.KernelDensityEstimation_tile(M.grid(ncols, nrows, 0.0, 0.0, cs, -9999.0), m)
    # the corners, the last rows and columns, and random cells
    rr = np.concatenate([[0, 0, nrows - 1, nrows - 1], r.integers(0, nrows, 260), np.full(40, nrows - 1)])
    cc = np.concatenate([[0, ncols - 1, 0, ncols - 1], r.integers(0, ncols, 260), r.integers(0, ncols, 40)])
    if m is not None:
        assert np.all(den[m == -9999.0] == -9999.0)
        keep = m[rr, cc] != -9999.0
        rr, cc = rr[keep], cc[keep]
    cx = ((cc + 0.5) * np.float64(np.float32(cs))).astype(np.float32)
    cy = ((nrows - 0.5 - rr) * np.float64(np.float32(cs))).astype(np.float32)
    h2 = (hs * hs).astype(np.float64)
    ref = want(x, y, w.astype(np.float64) / (h2 * TWO_PI_F), h2, cx, cy)
    tol = AMP * RTOL * ref.max() + 4.4e-9 * ref.max()
    assert np.all(np.abs(den[rr, cc] - ref) <= tol), np.max(np.abs(den[rr, cc] - ref)) / ref.max()


# 17M candidates and more: the split threshold is above 4096
@pytest.mark.parametrize("h_lo,h_hi", [(40.0, 60.0), (10.0, 80.0), (23.5, 25.0)])
@pytest.mark.parametrize("ncols,nrows", [(1024, 1024), (1025, 961)])
def test_wide_kernels(ctx, ncols, nrows, h_lo, h_hi):
    check(ctx, 400000 if h_hi > 30 else 800000, ncols, nrows, 1.0, h_lo, h_hi)


@pytest.mark.parametrize("cs", [0.3, 7.0])
def test_cell_size_and_mask(ctx, cs):
    check(ctx, 400000, 700, 900, cs, 20.0, 90.0, mask=True)


def test_tiles(ctx):
    """Tiles of 300 x 300: blocks of 44 columns or rows at their edges."""
    check(ctx, 400000, 900, 900, 1.0, 30.0, 70.0, tile=300)


def test_one_huge_bandwidth(ctx):
    """Every point inside the cut-off of every cell; few large blocks' worth of parts."""
    check(ctx, 120000, 1000, 800, 1.0, 2000.0, 3000.0)
