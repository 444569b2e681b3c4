"""Pilot densities and leave-one-out log-likelihoods where the branches of their
kernels meet: point counts around 16 and 64 queries and sums of 32, one to 17
candidates (a wave per candidate, candidates together, two passes), lists short
and long enough for each, crowded bins that are inside as a whole, waves that are
cut, duplicates and extreme weights.  Against sums in 64 bits over the pairs that
the exact cut-off predicate holds."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu
TWO_PI_F = np.float64(np.float32(6.2831853071795862))
EPS_DEN = np.float64(np.float32(1e-14))

# relative error of one density: 2^-24 for the rounding of the result, of a
# coefficient and of the exponent factor (times the exponent, at most 4.5), one
# rounding of the scaled exponent (at most 6.5 in base 2), about two of the
# exponential, 32 terms of a float sum and two of its Kahan pair
RTOL = (1 + 1 + 4.5 + 4.5 + 2 + 32 + 2) * 2.0 ** -24


def neighbours(x, y, h):
    """Ordered pairs (i, j), i != j, that may be within 3h, and their offsets."""
    p = np.stack([x, y], 1).astype(np.float64)
    ij = cKDTree(p).query_pairs(3.0 * h * (1 + 1e-5) + 1e-6, output_type="ndarray")
    i, j = np.concatenate([ij[:, 0], ij[:, 1]]), np.concatenate([ij[:, 1], ij[:, 0]])
    dx = (x[j] - x[i]).astype(np.float64)
    dy = (y[j] - y[i]).astype(np.float64)
    return i, j, dx * dx + dy * dy


def density(n, pairs, w, h, loo):
    i, j, d2 = pairs
    h2 = np.float64(np.float32(h) * np.float32(h))
    c = w.astype(np.float64) / (h2 * TWO_PI_F)
    k = np.where(d2 < 9.0 * h2, np.exp(d2 / (-2.0 * h2)) * c[j], 0.0)
    den = np.bincount(i, weights=k, minlength=n)
    return den if loo else den + c


def points(n, seed, crowd=0.0):
    """Clusters; the share `crowd` of the points in one spot of 2 x 2, a tenth of them twice."""
    r = np.random.default_rng(seed)
    k = r.integers(0, 5, n)
    x = (r.uniform(0, 400, 5)[k] + r.normal(0, 25, n)).astype(np.float32)
    y = (r.uniform(0, 400, 5)[k] + r.normal(0, 25, n)).astype(np.float32)
    m = int(crowd * n)
    x[:m] = (200 + r.uniform(0, 2, m)).astype(np.float32)
    y[:m] = (200 + r.uniform(0, 2, m)).astype(np.float32)
    d = m // 10
    x[d:2 * d], y[d:2 * d] = x[:d], y[:d]
    w = np.exp(r.normal(0, 3, n)).astype(np.float32)
    p = r.permutation(n)
    return x[p], y[p], w[p]


def check(ctx, x, y, w, hs):
    n = len(x)
    ctx.points_upload(x, y, w)
    pairs = neighbours(x, y, float(hs.max()))
    got = ctx.LogLikelihood(hs, edge_correction=False)
    for h, g in zip(hs, got):
        want = np.log(np.maximum(density(n, pairs, w, h, True), EPS_DEN)).sum()
        assert abs(g - want) <= n * RTOL * 1.001, (h, g, want)
    for h in (hs.min(), hs.max()):
        _, den0, _ = ctx.Abramson(float(h), 0.0, edge_correction=False)
        want = density(n, pairs, w, h, False)
        assert np.all(np.abs(den0 - want) <= RTOL * want)
        # the same estimator with a bandwidth per source (alpha = 0: all equal h)
        got = ctx.LogLikelihoodAdaptive([h], [0.0], edge_correction=False)[0]
        want = np.log(np.maximum(density(n, pairs, w, h, True), EPS_DEN)).sum()
        assert abs(got - want) <= n * RTOL * 1.001, (h, got, want)


@pytest.mark.parametrize("n", [2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 80, 129, 1000])
@pytest.mark.parametrize("k", [1, 2, 3, 17])
def test_counts(ctx, n, k):
    x, y, w = points(n, n + k)
    check(ctx, x, y, w, np.geomspace(2.0, 90.0, k).astype(np.float32))


@pytest.mark.parametrize("crowd", [0.3, 0.9])
@pytest.mark.parametrize("k", [2, 5])
def test_crowded_bins(ctx, crowd, k):
    """Bins of a thousand points, all inside for the largest bandwidths."""
    x, y, w = points(3000, 7, crowd)
    check(ctx, x, y, w, np.geomspace(0.05, 40.0, k).astype(np.float32))


@pytest.mark.parametrize("k", [2, 9, 16])
def test_long_lists(ctx, k):
    """16,500 points: candidates together from 16 of them on, and cut waves."""
    r = np.random.default_rng(3)
    x, y = r.uniform(0, 1000, (2, 16500)).astype(np.float32)
    x[:5000] = (500 + r.normal(0, 4, 5000)).astype(np.float32)
    w = np.exp(r.normal(0, 2, 16500)).astype(np.float32)
    check(ctx, x, y, w, np.geomspace(0.5, 22.0, k).astype(np.float32))
