"""Boundary distances where the search of a wave and the searches of its lanes meet:
few and many points on ragged, half ragged and smooth study areas, in clusters and
spread out, so that some waves search together, some lane by lane, and some give
the first up for the second.  Equal to brute force bit for bit, and not slow where
every cell of the raster is near a boundary."""
import time

import numpy as np
import pytest

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu


def area(kind, side, r):
    m = np.ones((side, side), np.float32)
    a = np.arange(side) - (side - 1) / 2
    if kind == "disk":
        m[a[:, None] ** 2 + a[None, :] ** 2 > (0.45 * side) ** 2] = -1
    elif kind == "dots":
        m[r.random((side, side)) < 0.02] = -1
    elif kind == "half":
        m[:, side // 2:][r.random((side, side - side // 2)) < 0.02] = -1
    elif kind == "coast":
        f = sum(np.interp(np.arange(side), np.linspace(0, side, 2 ** k + 1), r.normal(0, side * 0.25 / 2 ** k, 2 ** k + 1))
                for k in range(1, 9))
        m[np.arange(side)[None, :] < (side / 2 + f)[:, None]] = -1
    return m


def brute(x, y, flags):
    nr, nc = flags.shape
    r, c = np.nonzero(flags)
    cx, cy = (c + 0.5).astype(np.float32), (nr - 0.5 - r).astype(np.float32)
    out = np.empty(len(x))
    for k in range(len(x)):
        dx, dy = (cx - x[k]).astype(np.float64), (cy - y[k]).astype(np.float64)
        out[k] = (dx * dx + dy * dy).min()
    return out


@pytest.mark.parametrize("kind", ["disk", "dots", "half", "coast", "all"])
@pytest.mark.parametrize("n,clusters", [(64, 0), (700, 0), (700, 5)])
def test_equal_to_brute_force(ctx, kind, n, clusters):
    r = np.random.default_rng(n + clusters)
    side = 1100
    m = area(kind, side, r)
    if clusters:
        k = r.integers(0, clusters, n)
        x, y = (r.uniform(0, side, (2, clusters))[:, k] + r.normal(0, 4, (2, n))).astype(np.float32)
    else:
        x, y = r.uniform(-0.1 * side, 1.1 * side, (2, n)).astype(np.float32)
    ctx.points_upload(x, y)
    ctx.mask_upload(M.grid(side, side, 0.0, 0.0, 1.0, -1.0), m)
    d = ctx.CalcDist2Boundary()
    flags, _ = ctx.MarkBoundary()
    assert np.array_equal(d, brute(x, y, flags))


def test_few_points_on_a_ragged_area(ctx):
    """0.1 ms; 34 ms when a wave looked at all leaves around its points."""
    side = 8192
    r = np.random.default_rng(1)
    m = np.where(np.frombuffer(r.bytes(side * side), np.uint8).reshape(side, side) < 5, np.float32(-1), np.float32(1))
    ctx.mask_upload(M.grid(side, side, 0.0, 0.0, 1.0, -1.0), m)
    x, y = r.uniform(0, side, (2, 64)).astype(np.float32)
    ctx.points_upload(x, y)
    ctx.MarkBoundary()
    best = np.inf
    for _ in range(5):
        ctx.points_upload(x, y)
        ctx.synchronize()
        t = time.perf_counter()
        ctx.CalcDist2Boundary()
        best = min(best, time.perf_counter() - t)
    assert best < 10e-3
