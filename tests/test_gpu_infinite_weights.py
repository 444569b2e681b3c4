"""Infinite weights (an edge-correction weight is infinite where the kernel meets
no valid cell) in the sums that go through nodes of a block and moments of a
group, whose weights have both signs: a density is +inf inside the cut-off of such
a point and untouched outside, never NaN."""
import numpy as np
import pytest

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu
TWO_PI_F = np.float64(np.float32(6.2831853071795862))


def test_raster_everywhere_inside(ctx):
    """Every kernel covers every block and the blocks' wide kernels go to nodes."""
    r = np.random.default_rng(1)
    n, nc, nr = 120000, 1000, 800
    w = r.uniform(0.5, 2.0, n).astype(np.float32)
    w[777] = np.inf
    ctx.points_upload(r.uniform(0, nc, n).astype(np.float32), r.uniform(0, nr, n).astype(np.float32), w)
    ctx.set_bandwidths(r.uniform(2000, 3000, n).astype(np.float32))
    ctx.set_ec_weights(None)
    den = ctx.KernelDensityEstimation_tile(M.grid(nc, nr, 0.0, 0.0, 1.0, -9999.0))
    assert np.all(den == np.inf)


@pytest.mark.parametrize("target", [4096, 1024, 128])
def test_raster_blocks_in_and_out(target):
    """One infinite kernel of 60 cells: the blocks of 64 cells that it covers as a
    whole are +inf, those that it does not reach are as without it.  All points at
    the cells, at nodes in cut blocks, at nodes in whole blocks."""
    r = np.random.default_rng(2)
    n, side, h = 400000, 1024, 60.0
    x, y = r.uniform(0, side, (2, n)).astype(np.float32)
    w = r.uniform(0.5, 2.0, n).astype(np.float32)
    x[5], y[5] = 512.0, 512.0
    dens = []
    with M.Context(0) as ctx:
        ctx.set_option("density_split_target", target)
        for wt in (0.0, np.inf):
            w[5] = wt
            ctx.points_upload(x, y, w)
            ctx.set_bandwidth(h)
            ctx.set_ec_weights(None)
            dens.append(ctx.KernelDensityEstimation_tile(M.grid(side, side, 0.0, 0.0, 1.0, -9999.0)))
    c = np.arange(side) + 0.5
    lo, hi = c.reshape(-1, 64)[:, 0], c.reshape(-1, 64)[:, -1]
    far = np.maximum(np.abs(lo - 512), np.abs(hi - 512))
    near = np.maximum(0, np.maximum(lo - 512, 512 - hi))
    covered = far[:, None] ** 2 + far[None, :] ** 2 < (3 * h) ** 2
    reached = near[:, None] ** 2 + near[None, :] ** 2 < (3 * h) ** 2
    cells = lambda m: np.kron(m, np.ones((64, 64), bool))   # symmetric in x and y
    assert covered.sum() >= 4 and (~reached).sum() >= 100
    assert np.all(np.isfinite(dens[0]))
    assert np.all(dens[1][cells(covered)] == np.inf)
    assert np.array_equal(dens[1][~cells(reached)], dens[0][~cells(reached)])


@pytest.mark.parametrize("h", [2.0, 30.0, 400.0])
@pytest.mark.parametrize("loo", [True, False])
def test_points(ctx, h, loo):
    """Groups of 64 taken whole, some with an infinite member."""
    r = np.random.default_rng(3)
    n = 6000
    k = r.integers(0, 4, n)
    x = (r.uniform(0, 1000, 4)[k] + r.normal(0, 8, n)).astype(np.float32)
    y = (r.uniform(0, 1000, 4)[k] + r.normal(0, 8, n)).astype(np.float32)
    w = r.uniform(0.5, 2.0, n).astype(np.float32)
    w[[10, 2000, 2001]] = np.inf
    hs = r.uniform(h, 1.5 * h, n).astype(np.float32)
    ctx.points_upload(x, y, w)
    ctx.set_bandwidths(hs)
    ctx.set_ec_weights(None)
    got = ctx.DensityAtPoints(loo=loo).astype(np.float64)
    h2 = (hs * hs).astype(np.float64)
    ref = np.zeros(n)
    with np.errstate(invalid="ignore"):
        for i in range(0, n, 500):
            dx = (x[None, :] - x[i:i + 500, None]).astype(np.float64)
            dy = (y[None, :] - y[i:i + 500, None]).astype(np.float64)
            d2 = dx * dx + dy * dy
            t = np.exp(d2 / (-2.0 * h2)) / (h2 * TWO_PI_F) * w.astype(np.float64)
            t[d2 >= 9.0 * h2] = 0.0
            if loo:
                t[np.arange(len(d2)), i + np.arange(len(d2))] = 0.0
            ref[i:i + 500] = t.sum(1)
    assert np.array_equal(np.isinf(got), np.isinf(ref)) and not np.isnan(got).any()
    fin = np.isfinite(ref)
    assert 0 < fin.sum() < n or h > 300
    # the error bound of tests/test_gpu_fine_order.py: float chunks and truncated groups
    assert np.all(np.abs(got[fin] - ref[fin]) <= (77 * 2.0 ** -24 + 1.1e-8) * ref[fin])
