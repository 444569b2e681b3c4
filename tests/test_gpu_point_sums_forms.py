"""The forms of the leave-one-out sums against each other, and pairs that lie exactly on
the cut-off.  Candidates one by one (a wave per candidate, 16 or 64 queries), together
(k_loo_multi) and as a bandwidth per source give the same float sums: bit for bit where a
wave has the same 64 queries and is not cut (the places of the cuts follow from the largest
candidate), up to an ulp of a density where it has 16 (a bin that none of them reaches is
left out of the Kahan pair, which may then round a tie the other way).  On an integer lattice
with whole 3h every point has pairs at the cut-off."""
import numpy as np
import pytest

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu
TWO_PI_F = np.float64(np.float32(6.2831853071795862))
ULP = 2.0 ** -23   # of a density, relative
# the error bound of a density in tests/test_gpu_point_sums.py
RTOL = (1 + 1 + 4.5 + 4.5 + 2 + 32 + 2) * 2.0 ** -24


def loglik(ctx, hs):
    return ctx.LogLikelihood(np.asarray(hs, np.float32), edge_correction=False)


@pytest.mark.parametrize("n", [64, 700, 3000])
def test_few_points(ctx, n):
    """Sparse points with weights of very different sizes: one pair at the cut-off moves a
    density by 1e-3 and more."""
    r = np.random.default_rng(n)
    ctx.points_upload(*r.uniform(0, 30 * np.sqrt(n), (2, n)).astype(np.float32), np.exp(r.normal(0, 2, n)).astype(np.float32))
    hs = np.geomspace(12.0, 60.0, 16).astype(np.float32)
    alone = np.concatenate([loglik(ctx, [h]) for h in hs])
    assert np.array_equal(np.concatenate([loglik(ctx, hs[i:i + 2]) for i in range(0, 16, 2)]), alone)
    assert np.array_equal(loglik(ctx, hs), alone)          # one launch, a wave per candidate
    each = np.concatenate([ctx.LogLikelihoodAdaptive([h], [0.0], edge_correction=False) for h in hs])
    assert np.all(np.abs(each - alone) <= n * ULP)


def test_together_and_alone(ctx):
    """16,500 points: 16 candidates together, and one by one with 16 queries a wave."""
    r = np.random.default_rng(4)
    n = 16500
    x, y = (r.uniform(0, 1, (2, n)) * [[1000], [4000]]).astype(np.float32)
    ctx.points_upload(x, y, np.exp(r.normal(0, 2, n)).astype(np.float32))
    # at most 2,127 sources a wave, at the end of a row of bins: none is cut (4,096)
    hs = np.geomspace(6.0, 36.0, 16).astype(np.float32)
    alone = np.concatenate([loglik(ctx, [h]) for h in hs])
    assert np.all(np.abs(loglik(ctx, hs) - alone) <= n * ULP)


def test_together_and_alone_with_64_queries(ctx):
    """530,000 points along a line (a column of bins, so no wave spans a row and none is
    cut): one candidate alone takes 64 queries a wave, as three together do."""
    r = np.random.default_rng(5)
    n = 530000
    ctx.points_upload(r.uniform(0, 1, n).astype(np.float32), r.uniform(0, n, n).astype(np.float32),
                      np.exp(r.normal(0, 2, n)).astype(np.float32))
    hs = np.array([20.0, 45.0, 90.0], np.float32)
    assert np.array_equal(loglik(ctx, hs), np.concatenate([loglik(ctx, [h]) for h in hs]))


def lattice_loglik(side, h):
    """64 bits, exact cut-off fl64(d^2) < 9 fl32(h^2): sums over lattice offsets."""
    h2 = np.float64(np.float32(h) * np.float32(h))
    k = int(3 * h) + 2
    den = np.zeros((side, side))
    for dy in range(-k, k + 1):
        for dx in range(-k, k + 1):
            d2 = float(dx * dx + dy * dy)
            if (dx, dy) != (0, 0) and d2 < 9.0 * h2:
                den[max(0, dy):side + min(0, dy), max(0, dx):side + min(0, dx)] += np.exp(-d2 / (2 * h2))
    return np.log(den / (h2 * TWO_PI_F)).sum()


# 3h = 3, 4, 5, 6, 10: offsets (3, 0), (4, 0), (3, 4), (6, 0), (6, 8) at the cut-off
LATTICE = [1.0, 4.0 / 3.0, 5.0 / 3.0, 2.0, 10.0 / 3.0]


@pytest.mark.parametrize("side,k", [(24, 1), (24, 2), (24, 5), (131, 16)])
def test_lattice(ctx, side, k):
    """A pair more or less a point at the cut-off is 1e-4 to 2e-3 of a density, 40 times
    the tolerance and more over all points."""
    p = np.arange(side, dtype=np.float32)
    x, y = np.meshgrid(p, p)
    o = np.random.default_rng(side).permutation(side * side)
    ctx.points_upload(x.ravel()[o].copy(), y.ravel()[o].copy())
    n = side * side
    hs = np.array(LATTICE, np.float32)
    want = np.array([lattice_loglik(side, h) for h in hs])
    if k == 16:     # together: the lattice's candidates among others
        others = np.geomspace(0.9, 3.4, 11).astype(np.float32)
        got = loglik(ctx, np.concatenate([hs, others]))[:5]
    else:
        got = np.concatenate([loglik(ctx, hs[i:i + k]) for i in range(0, 5, k)])
    assert np.all(np.abs(got - want) <= n * RTOL * 1.001)
    each = np.concatenate([ctx.LogLikelihoodAdaptive([h], [0.0], edge_correction=False) for h in hs])
    assert np.all(np.abs(each - want) <= n * RTOL * 1.001)
