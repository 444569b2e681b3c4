"""Point densities in fine order (leave-one-out, a bandwidth per source) where
its branches meet: point counts around a group of 64, crowded bins whose groups
are taken whole, bandwidths from below the spacing to far above a group (every
class of group in one wave), duplicates, points without a bandwidth, and the
magnitudes at which a float distance over- or underflows.  Against the sum in
64 bits with the exact cut-off predicate."""
import numpy as np
import pytest

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu
TWO_PI_F = np.float64(np.float32(6.2831853071795862))

# relative error of one density: 2^-24 for the rounding of the result, of a
# coefficient and of the exponent factor (times the exponent, at most 4.5), one
# rounding of the scaled exponent (at most 6.5 in base 2) and about two of the
# exponential, and 64 terms of a float chunk: (1 + 1 + 4.5 + 4.5 + 2 + 64) 2^-24,
# and 1.1e-8 for the truncated group sums
RTOL = 77 * 2.0 ** -24 + 1.1e-8


def want(x, y, w, h, loo):
    h2 = (h * h).astype(np.float64)
    live = h2 > 0
    inv = np.where(live, h2, 1.0)
    out = np.zeros(len(x))
    for i in range(0, len(x), 512):
        dx = (x[None, :] - x[i:i + 512, None]).astype(np.float64)
        dy = (y[None, :] - y[i:i + 512, None]).astype(np.float64)
        d2 = dx * dx + dy * dy
        k = np.exp(d2 / (-2.0 * inv)) / (inv * TWO_PI_F) * w.astype(np.float64)
        k[(d2 >= 9.0 * h2) | ~live[None, :]] = 0.0
        if loo:
            k[np.arange(len(d2)), i + np.arange(len(d2))] = 0.0
        out[i:i + 512] = k.sum(1)
    return out


def check(ctx, x, y, w, h):
    ctx.points_upload(x, y, w)
    ctx.set_bandwidths(h)
    for loo in (True, False):
        got = ctx.DensityAtPoints(loo=loo).astype(np.float64)
        ref = want(x, y, w, h, loo)
        assert np.array_equal(got == 0, ref == 0)
        assert np.all(np.abs(got - ref) <= RTOL * ref)


def clustered(n, seed, spread):
    r = np.random.default_rng(seed)
    k = r.integers(0, 4, n)
    x = (r.uniform(0, 1000, 4)[k] + r.normal(0, spread, n)).astype(np.float32)
    y = (r.uniform(0, 1000, 4)[k] + r.normal(0, spread, n)).astype(np.float32)
    return x, y, r.uniform(0.5, 2.0, n).astype(np.float32), r


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 129, 1000, 5000])
@pytest.mark.parametrize("h", [0.05, 3.0, 60.0, 900.0])
def test_counts_and_bandwidths(ctx, n, h):
    x, y, w, r = clustered(n, n, 15.0)
    check(ctx, x, y, w, (h * np.exp(r.uniform(-0.3, 0.3, n))).astype(np.float32))


def test_every_class_in_a_wave(ctx):
    """Bandwidths over three decades in one crowded area."""
    x, y, w, r = clustered(6000, 7, 8.0)
    check(ctx, x, y, w, (10.0 ** r.uniform(-1.0, 2.0, 6000)).astype(np.float32))


def test_one_bandwidth_leave_one_out(ctx):
    x, y, w, r = clustered(4000, 9, 10.0)
    ctx.points_upload(x, y, w)
    ctx.set_bandwidth(40.0)
    h = np.full(4000, 40.0, np.float32)
    got = ctx.DensityAtPoints(loo=True).astype(np.float64)
    ref = want(x, y, w, h, True)
    assert np.all(np.abs(got - ref) <= RTOL * ref)


def test_duplicates_and_missing_bandwidths(ctx):
    r = np.random.default_rng(11)
    x = np.repeat(r.uniform(0, 50, 40), 50).astype(np.float32)
    y = np.repeat(r.uniform(0, 50, 40), 50).astype(np.float32)
    h = np.where(r.random(2000) < 0.3, 0.0, r.uniform(1.0, 20.0, 2000)).astype(np.float32)
    check(ctx, x, y, np.ones(2000, np.float32), h)


def test_cut_off_on_a_lattice(ctx):
    """Integer coordinates and 3h an integer: many pairs exactly at the cut-off."""
    g = np.arange(40, dtype=np.float32)
    x, y = (v.reshape(-1).copy() for v in np.meshgrid(g, g))
    check(ctx, x, y, np.ones(1600, np.float32), np.full(1600, 5.0, np.float32) / np.float32(3.0))
    check(ctx, x, y, np.ones(1600, np.float32), np.full(1600, 4.0, np.float32))


@pytest.mark.parametrize("scale", [1e-16, 1e12])
def test_magnitudes(ctx, scale):
    x, y, w, r = clustered(700, 13, 20.0)
    s = np.float32(scale)
    h = (25.0 * np.exp(r.uniform(-0.5, 0.5, 700))).astype(np.float32) * s
    ctx.points_upload(x * s, y * s, w)
    ctx.set_bandwidths(h)
    got = ctx.DensityAtPoints(loo=True).astype(np.float64)
    ref = want(x * s, y * s, w, h, True)
    assert np.all(np.abs(got - ref) <= RTOL * ref)
