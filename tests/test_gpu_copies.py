"""Copies between host and device of every size class: below one chunk, at the
chunk and lane edges, ragged tails, from one thread and from several contexts
at once.  An upload followed by a download is the identity on bytes."""
import threading

import numpy as np
import pytest

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu

CHUNK = 1 << 18   # floats of one pinned chunk (1 MB)


def round_trip(ctx, n, seed):
    """n bandwidths up, the same bandwidths back."""
    r = np.random.default_rng(seed)
    h = r.uniform(0.5, 2.0, n).astype(np.float32)
    x = r.uniform(0.0, 100.0, n).astype(np.float32)
    ctx.points_upload(x, x[::-1].copy())
    ctx.set_bandwidths(h)
    return np.array_equal(ctx.get_bandwidths(), h)


@pytest.mark.parametrize("n", [1, CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK + 7, 4 * CHUNK, 20 * CHUNK + 13])
def test_round_trip(ctx, n):
    assert round_trip(ctx, n, n)


def test_raster_comes_back_whole(ctx):
    """A 33 MB raster of nodata cells: every cell keeps its own mask value."""
    nr, nc = 2051, 4099
    mask = np.arange(nr * nc, dtype=np.float32).reshape(nr, nc)
    ctx.points_upload(np.array([5.0], np.float32), np.array([5.0], np.float32))
    ctx.set_bandwidth(0.25)
    den = ctx.KernelDensityEstimation_tile(M.grid(nc, nr, 0.0, 0.0, 1.0, -1.0), mask)
    assert den.shape == (nr, nc) and np.count_nonzero(den) <= 16
    got = ctx.KernelDensityEstimation_tile(M.grid(nc, nr, 1e6, 1e6, 1.0, float(mask[7, 9])), mask)
    assert got[7, 9] == mask[7, 9] and np.count_nonzero(got) == 1


def test_several_contexts_at_once():
    """More copies in flight than there are lanes."""
    ok = [False] * 4

    def work(i):
        with M.Context(0) as c:
            ok[i] = all(round_trip(c, 9 * CHUNK + 11 * i + k, 100 * i + k) for k in range(3))

    th = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert all(ok)
