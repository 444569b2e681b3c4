"""The check of uploaded coordinates (eight at a time): the first point that is not
finite is named at every place of a group of eight and in what is left over, a refused
upload leaves the earlier points usable, and the bounds count every point."""
import numpy as np
import pytest

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 9, 16, 1003])
def test_non_finite(ctx, n):
    ctx.points_upload(np.array([1, 2], np.float32), np.array([3, 4], np.float32))
    ctx.set_bandwidth(5.0)
    before = ctx.DensityAtPoints()
    for axis in (0, 1):
        for at in sorted({0, n // 2, n - 1}):
            for v in (np.nan, np.inf, -np.inf):
                p = np.full((2, n), 3e38, np.float32)
                p[axis, at:] = v
                with pytest.raises(M.MkdeError, match="point %d has a non-finite" % at):
                    ctx.points_upload(p[0], p[1])
    ctx.set_bandwidth(5.0)
    assert np.array_equal(ctx.DensityAtPoints(), before)


@pytest.mark.parametrize("n", [9, 100, 1003])
def test_bounds(ctx, n):
    """The extreme points are found by their neighbours, wherever they stand."""
    r = np.random.default_rng(n)
    for at in (0, 3, 8, n - 1):
        x, y = r.uniform(100, 200, (2, n)).astype(np.float32)
        x[at], y[at] = -5000.0, 7000.0
        x[(at + 1) % n], y[(at + 1) % n] = -5000.0, 7000.0
        ctx.points_upload(x, y)
        ctx.set_bandwidth(1.0)
        ctx.set_ec_weights(None)
        k = 1.0 / (2 * np.pi)
        d = ctx.DensityAtPoints(loo=True)
        assert abs(d[at] - k) < 1e-6 and abs(d[(at + 1) % n] - k) < 1e-6
