"""Node sums of the density raster where single points show: few thousand points a
block, so that each one near a cell is 1e-4 of it and more, against sums in 64 bits
with the exact cut-off, relative to the cell itself.  The split target decides whether
blocks are whole or cut and whether there are node sums at all; that they ran is seen
from the last bits, which the launch without a work list (all points at the cells) does
not share.  Bandwidths on both sides of the smallest that goes to the nodes, heavy
points at the places where parts are cut, rasters where some blocks have node sums and
others do not, ragged edges, tiles."""
import numpy as np
import pytest

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu
TWO_PI_F = np.float64(np.float32(6.2831853071795862))
RTOL = 1e-5   # what a density may be off, of itself


def want(x, y, coef, h2, cx, cy):
    out = np.zeros(len(cx))
    for i in range(0, len(cx), 64):
        dx = (cx[i:i + 64, None] - x[None, :]).astype(np.float64)
        dy = (cy[i:i + 64, None] - y[None, :]).astype(np.float64)
        d2 = dx * dx + dy * dy
        out[i:i + 64] = np.where(d2 < 9.0 * h2, np.exp(d2 / (-2.0 * h2)) * coef, 0.0).sum(1)
    return out


def rasters(x, y, w, h, nc, nr, target, tile=0):
    """The raster at this split target, and with all points at the cells."""
    with M.Context(0) as ctx:
        ctx.points_upload(x, y, w)
        ctx.set_bandwidths(h)
        ctx.set_ec_weights(None)
        out = []
        for order in (1, 0):
            ctx.set_option("density_order", order)
            ctx.set_option("density_split_target", target)
            if tile:
                out.append(ctx.KernelDensityEstimation_raster(nc, nr, [0.0, 1.0, 0.0, float(nr), 0.0, -1.0], -9999.0, tile, tile))
            else:
                out.append(ctx.KernelDensityEstimation_tile(M.grid(nc, nr, 0.0, 0.0, 1.0, -9999.0)))
        return out


def check(x, y, w, h, den, seed):
    """Two random cells of every block, and its corners."""
    r = np.random.default_rng(seed)
    nr, nc = den.shape
    rr, cc = [], []
    for a in range(0, nr, 64):
        for b in range(0, nc, 64):
            a1, b1 = min(a + 64, nr), min(b + 64, nc)
            rr += [a, a, a1 - 1, a1 - 1, *r.integers(a, a1, 2)]
            cc += [b, b1 - 1, b, b1 - 1, *r.integers(b, b1, 2)]
    rr, cc = np.array(rr), np.array(cc)
    if len(rr) > 900:
        k = r.choice(len(rr), 900, replace=False)
        rr, cc = rr[k], cc[k]
    h2 = (h * h).astype(np.float64)
    ref = want(x, y, w.astype(np.float64) / (h2 * TWO_PI_F), h2, (cc + 0.5).astype(np.float32), (nr - 0.5 - rr).astype(np.float32))
    e = np.abs(den[rr, cc] - ref)
    assert np.all(e <= RTOL * ref), np.max(e[ref > 0] / ref[ref > 0])


def points(n, nc, nr, h_lo, h_hi, seed):
    r = np.random.default_rng(seed)
    x, y = (r.uniform(0, 1, (2, n)) * [[nc], [nr]]).astype(np.float32)
    h = np.exp(r.uniform(np.log(h_lo), np.log(h_hi), n)).astype(np.float32)
    return x, y, r.uniform(0.5, 2.0, n).astype(np.float32), h, r


# Candidates of a block: about n (64 + 6 h)^2 / 1024^2, less at the edges; the split threshold is
# their sum over all blocks through the target, and from 4096 on there are node sums.  (Counted from
# the bins: thresholds of 4336 .. 6229 for cut blocks, half of them or all in 2 to 4 parts, and
# 17591 .. 49990 for whole ones, which none reaches.)
@pytest.mark.parametrize("nc,nr,tile", [(1024, 1024, 0), (1025, 961, 0), (900, 900, 300)])
@pytest.mark.parametrize("n,h_lo,h_hi,per", [(30000, 60.0, 60.0, 5500), (110000, 24.5, 26.0, 5500), (60000, 10.0, 80.0, 9000)])
@pytest.mark.parametrize("cut", [True, False])
def test_single_points(nc, nr, tile, n, h_lo, h_hi, per, cut):
    x, y, w, h, _ = points(n, nc, nr, h_lo, h_hi, n + nc)
    reach = 3 * h.max() + 1
    blocks = [(a, min(a + 63, (nc if not tile else tile * (1 + a // tile)) - 1)) for a in range(0, nc, 64)]
    total = n * len(blocks) * ((nr + 63) // 64) * (64 + 2 * reach) ** 2 / (nc * nr)
    # 64: the threshold is four times the average block
    den, plain = rasters(x, y, w, h, nc, nr, int(total / per) if cut else 64, tile)
    assert not np.array_equal(den, plain)   # some blocks went to the nodes
    assert np.all(np.abs(den.astype(np.float64) - plain) <= RTOL * plain)
    check(x, y, w, h, den, n)


@pytest.mark.parametrize("target", [64, 150, 330])
def test_heavy_points(target):
    """Every 97th point in bin order weighs a thousand times the others: wherever a
    part is cut, some stand at the cut."""
    x, y, w, h, r = points(30000, 1024, 1024, 24.3, 90.0, 5)
    order = np.lexsort((x // 47, y // 47))   # bins of 64 points, row by row
    w[order[::97]] *= 1000.0
    den, plain = rasters(x, y, w, h, 1024, 1024, target)
    assert not np.array_equal(den, plain)
    assert np.all(np.abs(den.astype(np.float64) - plain) <= RTOL * plain)
    check(x, y, w, h, den, target)


def test_some_blocks():
    """Wide kernels in the left half only: blocks that they do not reach keep their bits,
    and whole blocks with fewer than 192 of them too."""
    x, y, w, h, r = points(60000, 1024, 1024, 60.0, 60.0, 6)
    right = x > 300
    h[right] = 8.0
    den, plain = rasters(x, y, w, h, 1024, 1024, 64)
    far = slice(512, 1024)   # 300 + 180 and the next block's edge
    assert np.array_equal(den[:, far], plain[:, far])
    assert not np.array_equal(den[:, :256], plain[:, :256])
    check(x, y, w, h, den, 6)


def test_bandwidths_at_the_limit():
    """A block of 64 cells takes h >= 31.5 / 1.3 = 24.23 to the nodes: one bandwidth just
    above and one just below it give the same raster but for the rounding."""
    x, y, w, _, _ = points(110000, 1024, 1024, 1.0, 1.0, 7)
    dens = []
    for v in (24.22, 24.24):
        h = np.full(len(x), v, np.float32)
        den, plain = rasters(x, y, w, h, 1024, 1024, 64)
        assert np.array_equal(den, plain) == (v < 24.23)
        check(x, y, w, h, den, 7)
        dens.append(den)
