"""The allocation-free densities near the most points that fit the scratch array:
6.6M points that need few cut waves, in the orders that cut them most.  Equal to
the allocating entry point up to the order of the parts' sums."""
import numpy as np
import pytest

import mgpukde_tiled_amd as M
from test_zz_no_alloc import DeviceBuffer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,h,each,loo", [("uniform", 6_600_000, 0.5, True, False), ("uniform", 6_600_000, 0.5, True, True),
                                               ("clusters", 6_850_000, 2.0, False, True)])
def test_near_the_limit(kind, n, h, each, loo):
    r = np.random.default_rng(1)
    if kind == "uniform":
        x, y = r.uniform(0, 1e4, (2, n)).astype(np.float32)
    else:
        k = r.integers(0, 2000, n)
        x, y = (r.uniform(0, 1e4, (2, 2000))[:, k] + r.normal(0, 40, (2, n))).astype(np.float32)
    with M.Context(0) as ctx:
        ctx.points_upload(x, y)
        if each:
            ctx.set_bandwidths((h * np.exp(r.uniform(-0.7, 0.7, n))).astype(np.float32))
        else:
            ctx.set_bandwidth(h)
        ref = ctx.DensityAtPoints(loo=loo)
        buf = DeviceBuffer(4 * n)
        try:
            ctx.density_at_points_noalloc(loo, buf.ptr.value)
            got = buf.read(n)
        finally:
            buf.free()
    # waves may be cut at other places: 32 terms of a float sum either way
    assert np.all(np.abs(got - ref) <= 2 * 33 * 2.0 ** -24 * ref)
