"""Work lists of more units than one workgroup scans (16,384): density blocks and
64-query waves at the edges of a chunk of 4,096, with and without cut units, and a
search of that size through its captured graph.  Rasters against the launch without
a work list, densities against sums in 64 bits."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu
TWO_PI_F = np.float64(np.float32(6.2831853071795862))


@pytest.mark.parametrize("bx,by", [(128, 128), (113, 145), (160, 128), (241, 85), (227, 127)])
@pytest.mark.parametrize("crowd", [0, 60000])
def test_rasters(bx, by, crowd):
    """16,384 (one workgroup), 16,385, 20,480, 20,485 and 28,829 blocks; a crowd of points
    in one spot, whose blocks are cut."""
    r = np.random.default_rng(bx + crowd)
    nc, nr = 64 * bx - 5, 64 * by - 7
    x, y = (r.uniform(0, 1, (2, 3000 + crowd)) * [[nc], [nr]])
    if crowd:
        x[:crowd], y[:crowd] = nc * 0.7 + r.normal(0, 40, crowd), nr * 0.2 + r.normal(0, 40, crowd)
    with M.Context(0) as ctx:
        ctx.points_upload(x.astype(np.float32), y.astype(np.float32))
        ctx.set_bandwidth(9.0)
        ctx.set_ec_weights(None)
        g = M.grid(nc, nr, 0.0, 0.0, 1.0, -9999.0)
        den = ctx.KernelDensityEstimation_tile(g)
        ctx.set_option("density_order", 0)
        plain = ctx.KernelDensityEstimation_tile(g)
    if crowd:   # parts are added up in another order: 64 terms of a float sum
        assert np.all(np.abs(den - plain) <= 2 * 64 * 2.0 ** -24 * plain)
    else:
        assert np.array_equal(den, plain)


@pytest.mark.parametrize("waves", [16384, 16385, 20480, 20481])
@pytest.mark.parametrize("each", [False, True])
def test_points(waves, each):
    r = np.random.default_rng(waves)
    n, h = 64 * waves - 63 * (waves % 2), 6.0
    x, y = r.uniform(0, 8000, (2, n))
    x[:60000], y[:60000] = 3000 + r.normal(0, 30, 60000), 5000 + r.normal(0, 30, 60000)
    x, y = x.astype(np.float32), y.astype(np.float32)
    hs = (h * r.uniform(0.5, 1.0, n) if each else np.full(n, h)).astype(np.float32)
    with M.Context(0) as ctx:
        ctx.points_upload(x, y)
        if each:
            ctx.set_bandwidths(hs)
        else:
            ctx.set_bandwidth(h)
        ctx.set_ec_weights(None)
        got = ctx.DensityAtPoints(loo=False)
    assert np.all(got > 0)
    h2 = (hs * hs).astype(np.float64)
    q = np.concatenate([r.integers(0, 60000, 40), r.integers(60000, n, 400), [n - 1]])
    near = cKDTree(np.stack([x, y], 1)).query_ball_point(np.stack([x[q], y[q]], 1).astype(np.float64), 3.1 * h)
    for i, js in zip(q, near):
        js = np.asarray(js)
        d2 = (x[js] - x[i]).astype(np.float64) ** 2 + (y[js] - y[i]).astype(np.float64) ** 2
        ref = np.where(d2 < 9.0 * h2[js], np.exp(d2 / (-2.0 * h2[js])) / (h2[js] * TWO_PI_F), 0.0).sum()
        # the error bound of tests/test_gpu_fine_order.py
        assert abs(got[i] - ref) <= (77 * 2.0 ** -24 + 1.1e-8) * ref


def test_search_graph():
    """1.1M points: the captured search against the host-sized one, twice."""
    r = np.random.default_rng(7)
    n = 1_100_000
    x, y = r.uniform(0, 8000, (2, n)).astype(np.float32)
    hs = np.array([2.0, 3.0, 5.0], np.float32)
    with M.Context(0) as ctx:
        ctx.points_upload(x, y)
        graph = [ctx.LogLikelihood(hs, edge_correction=False) for _ in range(2)]
        ctx.set_option("search_graph", 0)
        host = ctx.LogLikelihood(hs, edge_correction=False)
    assert np.array_equal(graph[0], host) and np.array_equal(graph[1], host)
