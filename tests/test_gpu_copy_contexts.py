"""Large copies where contexts come and go or share the device: a context per call
does not pay for the copies of the ones before, a release gives the staging memory
back, and two jobs of a server whose rasters go through lanes at the same time come
out as alone."""
import time

import numpy as np
import pytest

import mgpukde_tiled_amd as M

pytestmark = pytest.mark.gpu


def call(side):
    """One raster from a context of its own: the raster and the time to destroy the context."""
    one = np.array([5.0], np.float32)
    c = M.Context(0)
    c.points_upload(one, one)
    c.set_bandwidth(0.5)
    c.set_ec_weights(None)
    d = c.KernelDensityEstimation_tile(M.grid(side, side, 0.0, 0.0, 1.0, -1.0))
    t = time.perf_counter()
    c.close()
    return d, time.perf_counter() - t


def test_a_context_per_call():
    """0.2 ms to destroy a context; 6.6 ms when its copies' streams went with it."""
    first, _ = call(2048)
    times = []
    for _ in range(9):
        d, t = call(2048)
        assert np.array_equal(d, first)
        times.append(t)
    assert np.median(times) < 3e-3


def test_release_and_copy_again():
    r = np.random.default_rng(1)
    h = r.uniform(1, 2, 4_000_000).astype(np.float32)
    x, y = r.uniform(0, 100, (2, len(h))).astype(np.float32)
    with M.Context(0) as c:
        for _ in range(3):
            c.points_upload(x, y)
            c.set_bandwidths(h)
            for _ in range(3):
                assert np.array_equal(c.get_bandwidths(), h)
            c.release()


def test_jobs_side_by_side():
    """Rasters of 33 MB from two slots: more than the least that lanes take there."""
    r = np.random.default_rng(2)
    nc, nr = 2900, 2903
    g = M.grid(nc, nr, 0.0, 0.0, 1.0, -9999.0)
    jobs = []
    for k in range(6):
        n = 3000 + 500 * k
        x, y = (r.uniform(0, 1, (2, n)) * [[nc], [nr]]).astype(np.float32)
        m = np.ones((nr, nc), np.float32)
        m[100 * k:100 * k + 700, 200:900] = -9999.0
        jobs.append((x, y, m))
    with M.Server(0, slots=2) as s:
        tickets = [s.submit(x, y, g, m, hoption=0) for x, y, m in jobs]
        got = []
        for t in tickets:
            res, den = s.wait(t)
            assert res["status"] == 0, res["message"]
            got.append(den)
    with M.Context(0) as c:
        for (x, y, m), den in zip(jobs, got):
            c.points_upload(x, y)
            c.mask_upload(g, m)
            c.tile_from_mask()
            c.run_job(hoption=0, optimise=False)
            assert np.array_equal(c.tile_download(), den)
