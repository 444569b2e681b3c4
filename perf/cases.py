"""Performance cases of mgpukde_tiled_amd: the calls a program makes, over their sizes.

A case is a dict of plain values.  `listed()` gives the named ones, `draw(rng)`
another of the same ranges, `prepare(case, seed)` the state a program holds
before the call, `run(state)` one pass through the public entry points with its
outputs, `work(case)` the bytes and floating-point operations of a pass that no
implementation can do without, and `exact(case, seed)` the outputs in 64 bits.

Kinds of call (`case["kind"]`):

  tile      edge-correction weights at given bandwidths (one value, or one per
            point), then the density raster of a tile
  raster    the density of a GeoTIFF-style raster of tiles at one bandwidth
  job       a whole job on resident inputs (boundary, edge correction,
            bandwidths, density raster), the raster copied out
  points    Abramson bandwidths, edge correction at them, leave-one-out
            densities at the points
  search    leave-one-out log-likelihoods of K fixed bandwidths
  adaptive  leave-one-out log-likelihoods of K (h, alpha) pairs of the adaptive
            estimator
  ingest    new points and a new mask on a context, boundary distances
  serve     a burst of mixed jobs through the job server, host data in and out
"""
import math

import numpy as np
import torch

import mgpukde_tiled_amd as M

NODATA = 0.0      # cells outside the study area, in the mask and in the raster that comes back
TWO_PI_F = float(np.float32(6.2831853071795862))   # the estimator's constant is a float
EPS_DEN = float(np.float32(1e-14))

# candidate bandwidths of a whole search span these multiples of the rule of
# thumb h; a golden-section step starts with two probes inside [h / 20, 2 h]
WIDE = (0.1, 10.0)
STEP = (0.6526, 1.3974)


# ------------------------------------------------------------------ inputs --
def _clip(v, extent):
    hi = np.nextafter(np.float32(extent), np.float32(0.0))
    return np.clip(v.astype(np.float32), np.float32(0.0), hi)


def _points(case, seed):
    """x, y, w (w is None where the case is unweighted) in [0, extent)^2."""
    r = np.random.default_rng(seed)
    n, ext = case["n"], _extent(case)
    how = case["points"]
    if how == "uniform":
        x, y = r.uniform(0.0, ext, n), r.uniform(0.0, ext, n)
    elif how == "thomas":      # clusters of about n / parents points, sigma 40 on an extent of 8192
        m = case["parents"]
        k = r.integers(0, m, n)
        s = ext * 40.0 / 8192.0
        x = r.uniform(0.0, ext, m)[k] + r.normal(0.0, s, n)
        y = r.uniform(0.0, ext, m)[k] + r.normal(0.0, s, n)
    elif how == "mixture":     # half uniform, half in 64 clusters of sigma 2% of the extent
        k = r.integers(0, 64, n - n // 2)
        cx, cy = r.uniform(0.0, ext, 64), r.uniform(0.0, ext, 64)
        x = np.concatenate([r.uniform(0.0, ext, n // 2), cx[k] + r.normal(0.0, 0.02 * ext, len(k))])
        y = np.concatenate([r.uniform(0.0, ext, n // 2), cy[k] + r.normal(0.0, 0.02 * ext, len(k))])
    else:                      # lognormal: cluster intensities lognormal (sigma 1.5), offsets N(0, 64 cells)
        m = case["parents"]
        lam = r.lognormal(0.0, 1.5, m)
        k = np.repeat(np.arange(m), r.multinomial(n, lam / lam.sum()))
        s = 64.0 * case["cs"]
        x = r.uniform(0.0, ext, m)[k] + r.normal(0.0, s, n)
        y = r.uniform(0.0, ext, m)[k] + r.normal(0.0, s, n)
    w = r.uniform(0.5, 2.0, n).astype(np.float32) if case["weights"] else None
    return _clip(x, ext), _clip(y, ext), w


def _extent(case):
    return float(case["cs"]) * max(case["ncols"], case["nrows"])


def _mask(case, seed, ncols=None, nrows=None):
    """Mask values: a disk or a rectangle of valid cells minus holes, or all valid."""
    ncols, nrows = ncols or case["ncols"], nrows or case["nrows"]
    r = np.random.default_rng(seed + 1000)
    if case["mask"] == "all":
        return np.ones((nrows, ncols), np.float32)
    m = np.full((nrows, ncols), NODATA, np.float32)
    if case["mask"] == "disk":
        rad = 0.476 * min(ncols, nrows)
        dy = np.arange(nrows) - (nrows - 1) / 2.0
        half = np.sqrt(np.maximum(rad * rad - dy * dy, 0.0))
        lo = np.ceil((ncols - 1) / 2.0 - half).astype(int)
        hi = np.floor((ncols - 1) / 2.0 + half).astype(int)
        for i in np.flatnonzero(np.abs(dy) <= rad):
            m[i, max(lo[i], 0):hi[i] + 1] = 1.0
    else:
        w, h = max(1, int(ncols * r.uniform(0.6, 0.9))), max(1, int(nrows * r.uniform(0.6, 0.9)))
        m[(nrows - h) // 2:(nrows - h) // 2 + h, (ncols - w) // 2:(ncols - w) // 2 + w] = 1.0
    for _ in range(case["holes"]):
        side = max(3, min(ncols, nrows) // 20)
        hw, hh = int(r.integers(2, side + 1)), int(r.integers(2, side + 1))
        c0, r0 = int(r.integers(0, max(1, ncols - hw))), int(r.integers(0, max(1, nrows - hh)))
        m[r0:r0 + hh, c0:c0 + hw] = NODATA
    return m


def _grid(case):
    return M.grid(case["ncols"], case["nrows"], 0.0, 0.0, case["cs"], NODATA)


def _rule(x, y, w):
    """The rule-of-thumb bandwidth with the estimator's float sums in point order."""
    w = np.ones(len(x), np.float32) if w is None else w
    sw = np.cumsum(w, dtype=np.float32)[-1]
    mx = np.cumsum(w * x, dtype=np.float32)[-1] / sw
    my = np.cumsum(w * y, dtype=np.float32)[-1] / sw
    d2 = (x - mx).astype(np.float64) ** 2 + (y - my).astype(np.float64) ** 2
    d2 = float((w.astype(np.float64) * d2).sum() / w.astype(np.float64).sum())
    return np.sqrt(np.float32(float(np.sqrt(np.float32(2.0) / np.float32(3 * len(x)))) * d2))


def _candidates(h0, k, lo=WIDE[0], hi=WIDE[1]):
    t = np.arange(k) / max(k - 1, 1)
    return (float(h0) * lo * (hi / lo) ** t).astype(np.float32)


def _bandwidths(case, x, y, w, seed):
    """The bandwidths a tile case is given: one value (a share of the rule of
    thumb), or one per point spread over a factor of six as a file of adaptive
    bandwidths holds them."""
    h0 = float(_rule(x, y, w)) * case["h"]
    if not case["per_point"]:
        return np.float32(h0)
    r = np.random.default_rng(seed + 2000)
    return (h0 * np.exp(r.uniform(-0.9, 0.9, len(x)))).astype(np.float32)


def _serve_jobs(case, seed):
    """The burst of a serve case: points log-uniform, uniform or clustered,
    square rasters with log-uniform sides, half rule of thumb, 30% adaptive,
    20% searches over 16 candidates."""
    r = np.random.default_rng(case["mix"])     # the sizes are the case's, the data the seed's
    jobs = []
    for i in range(case["jobs"]):
        n = int(round(math.exp(r.uniform(math.log(case["n_lo"]), math.log(case["n_hi"])))))
        side = int(round(math.exp(r.uniform(math.log(case["side_lo"]), math.log(case["side_hi"])))))
        u = r.random()
        j = {"n": n, "ncols": side, "nrows": side, "cs": 1.0, "weights": False, "holes": int(r.integers(0, 8)),
             "points": "thomas" if r.random() < 0.5 else "uniform", "parents": max(1, n // 500),
             "mask": "disk" if r.random() < 0.5 else "rect", "hoption": 0 if u < 0.5 else (2 if u < 0.8 else 3)}
        x, y, _ = _points(j, seed + 7 * i)
        jobs.append((j, x, y, _mask(j, seed + 7 * i)))
    return jobs


# ------------------------------------------------------------------- cases --
def _case(kind, **kw):
    c = {"kind": kind, "weights": False, "holes": 0, "mask": "all", "parents": 1, "points": "uniform", "cs": 1.0}
    c.update(kw)
    return c


def listed():
    return [
        # the generated-points mode: 100 points, a 1000 x 1000 tile; launches and waits count
        _case("tile", name="tile_100", n=100, ncols=1000, nrows=1000, cs=0.1, h=1.0, per_point=False, ec_cells=100),
        # bandwidths read from a file, a ragged masked raster with coarse cells
        _case("tile", name="tile_file_60k", n=60013, ncols=3001, nrows=1777, cs=2.5, h=0.3, per_point=True, ec_cells=0,
              points="thomas", parents=150, weights=True, mask="rect", holes=7),
        # a raster of GeoTIFF tiles at a small bandwidth: the density of a 10M-point, 32768^2 raster
        _case("raster", name="raster_h16", n=625000, ncols=8192, nrows=8192, tile=4096, h=16.0, points="lognormal",
              parents=64),
        # the headline job: 1M clustered, weighted points, adaptive bandwidths, edge corrected, 8192^2
        _case("job", name="job_1m", n=1000000, ncols=8192, nrows=8192, hoption=2, points="thomas", parents=200,
              weights=True, mask="disk", holes=20),
        # an everyday job: rule-of-thumb bandwidth, a raster of ordinary size
        _case("job", name="job_fixed_50k", n=50000, ncols=1500, nrows=1200, hoption=0, points="mixture", mask="disk",
              holes=5),
        # the estimate at the points only (no raster): adaptive bandwidths and cross-validated densities
        _case("points", name="points_1m", n=1000000, ncols=8192, nrows=8192, points="thomas", parents=200,
              weights=True, mask="disk", holes=20),
        # the batched bandwidth search: 64 candidates
        _case("search", name="search_64", n=200000, ncols=4096, nrows=4096, k=64, points="mixture", lo=WIDE[0],
              hi=WIDE[1]),
        # one step of the golden-section optimiser: two candidates, called again and again
        _case("search", name="search_2", n=100000, ncols=2048, nrows=2048, k=2, points="thomas", parents=100,
              mask="disk", holes=6, lo=STEP[0], hi=STEP[1]),
        # one probe of the (h, alpha) optimiser
        _case("adaptive", name="adaptive_2", n=100000, ncols=2048, nrows=2048, k=2, points="thomas", parents=100,
              weights=True, mask="disk", holes=6),
        # new data on a context that is kept
        _case("ingest", name="ingest_1m", n=1000000, ncols=4096, nrows=4096, points="thomas", parents=200,
              weights=True, mask="disk", holes=20),
        # one small request to the job server
        _case("serve", name="serve_1", jobs=1, mix=3, n_lo=2000, n_hi=2001, side_lo=300, side_hi=301),
        # a burst of mixed requests
        _case("serve", name="serve_16", jobs=16, mix=5, n_lo=1000, n_hi=300000, side_lo=256, side_hi=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tile", "raster", "job", "points", "search", "adaptive", "ingest", "serve"])
    how = rng.choice(["uniform", "thomas", "mixture", "lognormal"])
    mask = rng.choice(["disk", "rect", "all"])
    kw = {"points": how, "parents": _log_int(rng, 8, 200), "weights": rng.random() < 0.5, "mask": mask,
          "holes": rng.randrange(0, 12), "cs": rng.choice([1.0, 1.0, 0.5, 2.5])}
    if kind == "tile":
        kw.update(n=_log_int(rng, 50, 60000), ncols=_log_int(rng, 200, 3000), nrows=_log_int(rng, 200, 3000),
                  h=rng.uniform(0.15, 1.0), per_point=rng.random() < 0.5, ec_cells=0)
    elif kind == "raster":
        kw.update(n=_log_int(rng, 10000, 600000), ncols=_log_int(rng, 1000, 8000), nrows=_log_int(rng, 1000, 8000),
                  tile=rng.choice([1000, 2048, 4096]), cs=1.0, h=rng.uniform(6.0, 24.0))
    elif kind == "job":
        side = _log_int(rng, 300, 4000)
        kw.update(n=_log_int(rng, 1000, 250000), ncols=side, nrows=max(200, int(side * rng.uniform(0.6, 1.0))),
                  hoption=rng.choice([0, 2]))
    elif kind == "points":
        side = _log_int(rng, 500, 8000)
        kw.update(n=_log_int(rng, 2000, 800000), ncols=side, nrows=max(200, int(side * rng.uniform(0.6, 1.0))))
    elif kind == "search":
        lo, hi = rng.choice([WIDE, STEP])
        k = rng.randrange(1, 49) if hi > 2.0 else rng.randrange(1, 9)
        kw.update(n=_log_int(rng, 2000, 100000), ncols=_log_int(rng, 300, 3000), nrows=_log_int(rng, 300, 3000), k=k,
                  lo=lo, hi=hi)
    elif kind == "adaptive":
        kw.update(n=_log_int(rng, 2000, 150000), ncols=_log_int(rng, 300, 3000), nrows=_log_int(rng, 300, 3000),
                  k=rng.randrange(1, 5))
    elif kind == "ingest":
        kw.update(n=_log_int(rng, 1000, 1000000), ncols=_log_int(rng, 300, 4000), nrows=_log_int(rng, 300, 4000))
    else:
        return _case("serve", jobs=rng.randrange(1, 13), mix=rng.randrange(1 << 30), n_lo=1000,
                     n_hi=_log_int(rng, 3000, 200000), side_lo=256, side_hi=_log_int(rng, 400, 2048))
    return _case(kind, **kw)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        jobs = []
        for j, x, y, m in _serve_jobs(case, seed):
            jobs.append((x, y, M.grid(j["ncols"], j["nrows"], 0.0, 0.0, 1.0, NODATA), m, j["hoption"]))
        return {"case": case, "server": M.Server(slots=4), "jobs": jobs}
    x, y, w = _points(case, seed)
    ctx = M.Context(0)
    st = {"case": case, "ctx": ctx}
    if kind == "ingest":
        st.update(x=x, y=y, w=w, grid=_grid(case), mask=_mask(case, seed))
        return st
    ctx.points_upload(x, y, w)
    if kind == "tile":
        if case["ec_cells"]:
            k = case["ec_cells"]
            ctx.mask_upload(M.grid(k, k, 0.0, 0.0, _extent(case) / k, NODATA), np.ones((k, k), np.float32))
            st["tile_mask"] = None
        else:
            st["tile_mask"] = _mask(case, seed)
            ctx.mask_upload(_grid(case), st["tile_mask"])
        st.update(grid=_grid(case), h=_bandwidths(case, x, y, w, seed))
    elif kind == "raster":
        ctx.set_bandwidth(case["h"])
        ctx.set_ec_weights(None)
        e = _extent(case)
        st["gt"] = [0.0, case["cs"], 0.0, e, 0.0, -case["cs"]]
    else:
        ctx.mask_upload(_grid(case), _mask(case, seed))
        if kind == "job":
            ctx.tile_from_mask()
        elif kind == "points":
            st["h0"] = float(_rule(x, y, w))
        elif kind == "search":
            st["h"] = _candidates(_rule(x, y, w), case["k"], case["lo"], case["hi"])
        elif kind == "adaptive":
            st["h"], st["alpha"] = _pairs(case, float(_rule(x, y, w)))
    return st


def _pairs(case, h0):
    k = np.arange(case["k"])
    return (h0 * (1.0 - 0.1 * k)).astype(np.float32), (-0.5 + 0.1 * (k % 2)).astype(np.float32)


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "serve":
        srv = st["server"]
        tickets = [srv.submit(x, y, g, m, hoption=ho) for x, y, g, m, ho in st["jobs"]]
        out = []
        for t in tickets:
            r, raster = srv.wait(t)
            if r["status"] != 0:
                raise RuntimeError(r["message"])
            out.append((raster, np.float32(r["h_sel"])))
        return out
    ctx = st["ctx"]
    if kind == "ingest":
        ctx.points_upload(st["x"], st["y"], st["w"])
        ctx.mask_upload(st["grid"], st["mask"])
        return ctx.CalcDist2Boundary()
    if kind == "tile":
        if case["per_point"]:
            ctx.set_bandwidths(st["h"])
        else:
            ctx.set_bandwidth(st["h"])
        ew, pairs = ctx.EdgeCorrectionWeightsExact()
        return {"ew": ew, "pairs": pairs, "density": ctx.KernelDensityEstimation_tile(st["grid"], st["tile_mask"])}
    if kind == "raster":
        return ctx.KernelDensityEstimation_raster(case["ncols"], case["nrows"], st["gt"], NODATA, case["tile"],
                                                  case["tile"])
    if kind == "job":
        s = ctx.run_job(hoption=case["hoption"], optimise=False)
        return {"density": ctx.tile_download(), "h": ctx.get_bandwidths(), "ew": ctx.get_ec_weights(),
                "pairs": s["n_ec_pairs"]}
    if kind == "points":
        h, den0, g = ctx.Abramson(st["h0"])
        ew, pairs = ctx.EdgeCorrectionWeightsExact()
        return {"h": h, "den0": den0, "ew": ew, "pairs": pairs, "den1": ctx.DensityAtPoints(loo=True)}
    if kind == "search":
        return ctx.LogLikelihood(st["h"])
    return ctx.LogLikelihoodAdaptive(st["h"], st["alpha"])


# ---------------------------------------------------------- least work -----
def _typical_h(case, n):
    """The rule-of-thumb bandwidth of points spread evenly over the extent."""
    e = _extent(case)
    return math.sqrt(math.sqrt(2.0 / (3.0 * n)) * e * e / 6.0)


def _job_work(n, cells, h, cs, hoption, k):
    """(bytes, flops): inputs and outputs once; one multiply-add per (point,
    cell) pair inside the cut-off of 3h on the raster, ten operations per
    (point, point) pair, the cells of a row summed once in edge correction."""
    area = math.pi * (3.0 * h / cs) ** 2
    share = min(1.0, area / max(cells, 1))
    b = 12.0 * n + 8.0 * cells
    f = 2.0 * n * min(area, cells) + n * 40.0 * 6.0 * h / cs
    if hoption in (2, 3):
        f += 10.0 * k * n * n * share
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "serve":
        b = f = 0.0
        r = np.random.default_rng(case["mix"])
        for i in range(case["jobs"]):
            n = int(round(math.exp(r.uniform(math.log(case["n_lo"]), math.log(case["n_hi"])))))
            side = int(round(math.exp(r.uniform(math.log(case["side_lo"]), math.log(case["side_hi"])))))
            u = r.random()
            r.integers(0, 8), r.random(), r.random()
            ho = 0 if u < 0.5 else (2 if u < 0.8 else 3)
            w = _job_work(n, side * side, math.sqrt(math.sqrt(2.0 / (3.0 * n)) / 6.0) * side, 1.0, ho,
                          16 if ho == 3 else 1)
            b, f = b + w[0], f + w[1]
        return {"bytes": b, "flops": f}
    n, cells, cs = case["n"], case["ncols"] * case["nrows"], case["cs"]
    h = _typical_h(case, n)
    cols = 6.0 * h / cs
    if kind == "ingest":
        return {"bytes": 20.0 * n + 4.0 * cells, "flops": 10.0 * n}
    if kind == "tile":
        b, f = _job_work(n, cells, h * case["h"], cs, 0, 1)
        return {"bytes": b + 8.0 * n, "flops": f}
    if kind == "raster":
        return {"bytes": 12.0 * n + 4.0 * cells, "flops": 2.0 * n * math.pi * (3.0 * case["h"] / cs) ** 2}
    if kind == "job":
        b, f = _job_work(n, cells, h, cs, case["hoption"], 1)
        return {"bytes": b + 8.0 * n, "flops": f}
    pair = 10.0 * n * n * min(1.0, math.pi * (3.0 * h) ** 2 / (cells * cs * cs))
    if kind == "points":
        return {"bytes": 28.0 * n + cells, "flops": 2.0 * pair + 2.0 * n * 40.0 * cols}
    if kind == "adaptive":
        return {"bytes": case["k"] * 12.0 * n + cells, "flops": case["k"] * (2.0 * pair + 2.0 * n * 40.0 * cols)}
    f = 0.0
    for hk in _candidates(h, case["k"], case["lo"], case["hi"]).astype(float):
        share = min(1.0, math.pi * (3.0 * hk) ** 2 / (cells * cs * cs))
        f += 10.0 * n * n * share + n * 40.0 * min(6.0 * hk / cs, case["ncols"])
    return {"bytes": 12.0 * n + cells + 8.0 * case["k"], "flops": float(f)}


# ------------------------------------------------------- 64-bit results ----
# Most (query, source) pairs looked at in one 64-bit evaluation (about 20 s)
EXACT_PAIRS = 7e11


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a, dtype=None):
    return torch.as_tensor(np.ascontiguousarray(a), device=_dev(), dtype=dtype)


class _Budget:
    """Counts the pairs looked at; False once an evaluation has grown too large."""

    def __init__(self, left=EXACT_PAIRS):
        self.left = left

    def take(self, pairs):
        self.left -= pairs
        return self.left >= 0


def _centres(ncols, nrows, xll, yll, cs):
    cx = (np.float64(xll) + (np.arange(ncols) + 0.5) * np.float64(cs)).astype(np.float32)
    cy = (np.float64(yll) + (np.float64(nrows) - 0.5 - np.arange(nrows)) * np.float64(cs)).astype(np.float32)
    return cx, cy


def _h2(h):
    """The estimator's squared bandwidth: a float product, then 64 bits."""
    return (h * h).double()


def _kernel_sum(qx, qy, sx, sy, coef, h2, self_at=None):
    """sum over sources of coef exp(-d2 / 2 h2) inside d2 < 9 h2, for float
    coordinates, in chunks; self_at: the source index of query 0 (left out)."""
    out = torch.zeros(len(qx), dtype=torch.float64, device=qx.device)
    step = max(1, (1 << 25) // max(1, len(qx)))
    for s in range(0, len(sx), step):
        e = min(len(sx), s + step)
        d2 = (sx[None, s:e] - qx[:, None]).double().square_()
        d2 += (sy[None, s:e] - qy[:, None]).double().square_()
        v = torch.exp(d2 / (-2.0 * h2[None, s:e]))
        v *= coef[None, s:e]
        v.masked_fill_(d2 >= 9.0 * h2[None, s:e], 0.0)
        if self_at is not None:
            v.masked_fill_(self_at[:, None] == torch.arange(s, e, device=qx.device)[None, :], 0.0)
        out += v.sum(1)
    return out


def _near(sx, sy, h2, x0, x1, y0, y1):
    """Sources whose cut-off may reach a box."""
    gx = (torch.clamp(x0 - sx, min=0) + torch.clamp(sx - x1, min=0)).double()
    gy = (torch.clamp(y0 - sy, min=0) + torch.clamp(sy - y1, min=0)).double()
    return torch.nonzero(gx * gx + gy * gy < 9.0 * h2 * 1.00001).reshape(-1)


def _point_density(x, y, coef, h2, loo, bud):
    """Density at every point, boxes of neighbouring points at a time."""
    n = len(x)
    ext = float(max(x.max() - x.min(), y.max() - y.min(), torch.tensor(1e-6)))
    k = max(1, min(64, int(math.sqrt(n / 256))))
    b = ((x - x.min()) / ext * k).long().clamp(max=k - 1) * k + ((y - y.min()) / ext * k).long().clamp(max=k - 1)
    order = torch.argsort(b)
    cnt = torch.bincount(b, minlength=k * k).tolist()
    out = torch.zeros(n, dtype=torch.float64, device=x.device)
    at = 0
    for c in cnt:
        if not c:
            continue
        for s in range(0, c, 8192):
            q = order[at + s:at + min(c, s + 8192)]
            qx, qy = x[q], y[q]
            near = _near(x, y, h2, qx.min(), qx.max(), qy.min(), qy.max())
            if not bud.take(len(q) * len(near)):
                return None
            self_at = torch.searchsorted(near, q) if loo else None
            out[q] = _kernel_sum(qx, qy, x[near], y[near], coef[near], h2[near], self_at)
        at += c
    return out


def _boundary_dist(x, y, mask, cx, cy):
    v = mask != NODATA
    p = torch.zeros((v.shape[0] + 2, v.shape[1] + 2), dtype=torch.bool, device=v.device)
    p[1:-1, 1:-1] = v
    inner = torch.ones_like(v)
    for dr in range(3):
        for dc in range(3):
            inner &= p[dr:dr + v.shape[0], dc:dc + v.shape[1]]
    rr, cc = torch.nonzero(v & ~inner, as_tuple=True)
    bx, by = cx[cc], cy[rr]
    out = torch.full((len(x),), torch.finfo(torch.float64).max, dtype=torch.float64, device=x.device)
    step = max(1, (1 << 25) // max(1, len(bx)))
    for s in range(0, len(x), step):
        d2 = (bx[None] - x[s:s + step, None]).double().square_()
        d2 += (by[None] - y[s:s + step, None]).double().square_()
        if d2.shape[1]:
            out[s:s + step] = d2.min(1).values
    return out


def _ec(x, y, h, mask, cx, cy, cs, dist, bud):
    """Edge-correction weights and the number of cells inside the cut-offs."""
    ew = torch.ones(len(x), dtype=torch.float64, device=x.device)
    h2 = _h2(h)
    act = torch.nonzero(dist < 9.0 * h2).reshape(-1)
    box = max(float((3.0 * h[act]).median()) if len(act) else 1.0, 4.0 * cs)
    act = act[torch.argsort((y[act] / box).floor().long() * (1 << 20) + (x[act] / box).floor().long())]
    valid = mask != NODATA
    total = 0
    for s in range(0, len(act), 64):
        p = act[s:s + 64]
        r = 3.0 * h[p].double() + cs
        rows = (cy.double() >= (y[p].double() - r).min()) & (cy.double() <= (y[p].double() + r).max())
        cols = (cx.double() >= (x[p].double() - r).min()) & (cx.double() <= (x[p].double() + r).max())
        rows, cols = torch.nonzero(rows).reshape(-1).cpu(), torch.nonzero(cols).reshape(-1).cpu()
        if not len(rows) or not len(cols):
            ew[p] = float("inf")
            continue
        r0, r1, c0, c1 = int(rows[0]), int(rows[-1]) + 1, int(cols[0]), int(cols[-1]) + 1
        if not bud.take(len(p) * (r1 - r0) * (c1 - c0)):
            return None, 0
        dx2 = (cx[None, c0:c1] - x[p, None]).double().square_()
        ex = torch.exp(dx2 / (-2.0 * h2[p, None]))
        acc = torch.zeros(len(p), dtype=torch.float64, device=x.device)
        step = max(1, (1 << 25) // (len(p) * (c1 - c0)))
        for a in range(r0, r1, step):
            b = min(r1, a + step)
            dy2 = (cy[None, a:b] - y[p, None]).double().square_()
            ey = torch.exp(dy2 / (-2.0 * h2[p, None]))
            ins = (dx2[:, None, :] + dy2[:, :, None] < 9.0 * h2[p, None, None]) & valid[None, a:b, c0:c1]
            total += int(ins.sum())
            acc += ((ins * ex[:, None, :]).sum(2) * ey).sum(1)
        area = float(np.float32(cs) * np.float32(cs))
        ew[p] = 1.0 / (acc * area / (h2[p] * TWO_PI_F))
    return ew, total


def _cells(x, y, coef, h2, cx, cy, bud):
    """Density at cells cy x cx, 64 x 128 cells at a time."""
    out = torch.zeros((len(cy), len(cx)), dtype=torch.float64, device=x.device)
    for r in range(0, len(cy), 64):
        ys = cy[r:r + 64]
        band = torch.nonzero((torch.clamp(ys.min() - y, min=0) + torch.clamp(y - ys.max(), min=0)).double().square()
                             < 9.0 * h2 * 1.00001).reshape(-1)
        bx, by, bh, bc = x[band], y[band], h2[band], coef[band]
        for c in range(0, len(cx), 128):
            xs = cx[c:c + 128]
            near = _near(bx, by, bh, xs.min(), xs.max(), ys.min(), ys.max())
            if not bud.take(len(near) * len(xs) * len(ys)):
                return None
            for s in range(0, len(near), 4096):
                i = near[s:s + 4096]
                dx2 = (xs[None] - bx[i, None]).double().square_()
                dy2 = (ys[None] - by[i, None]).double().square_()
                k = torch.exp(dx2 / (-2.0 * bh[i, None]))[:, None, :] \
                    * (torch.exp(dy2 / (-2.0 * bh[i, None])) * bc[i, None])[:, :, None]
                k.masked_fill_(dx2[:, None, :] + dy2[:, :, None] >= 9.0 * bh[i, None, None], 0.0)
                out[r:r + 64, c:c + 128] += k.sum(0)
    return out


def _coef(w, ew, h2):
    return w.double() * ew / (h2 * TWO_PI_F)


def _adapt(x, y, w, h0, alpha, mask, cx, cy, cs, dist, bud):
    """Pilot densities at h0 and the adaptive bandwidths (floats) that follow."""
    hh = torch.full_like(x, float(h0))
    ew, _ = _ec(x, y, hh, mask, cx, cy, cs, dist, bud)
    den0 = None if ew is None else _point_density(x, y, _coef(w, ew, _h2(hh)), _h2(hh), False, bud)
    if den0 is None:
        return None, None
    g = torch.exp(torch.log(den0).mean())
    return den0, (float(h0) * (den0 / g) ** float(alpha)).float()


def _raster(out, mask):
    if mask is not None:
        out = torch.where(mask != NODATA, out, mask.double())
    return out.cpu().numpy()


def _exact_job(case, x, y, w, mask, hoption, bud):
    """density, h, ew, pairs of a job; None where it would take too long."""
    h0 = _rule(x, y, w)
    wt = _t(np.ones(len(x), np.float32) if w is None else w)
    x, y, m = _t(x), _t(y), _t(mask)
    cxn, cyn = _centres(case["ncols"], case["nrows"], 0.0, 0.0, case["cs"])
    cx, cy = _t(cxn), _t(cyn)
    dist = _boundary_dist(x, y, m, cx, cy)
    if hoption == 2:
        _, h = _adapt(x, y, wt, h0, -0.5, m, cx, cy, case["cs"], dist, bud)
        if h is None:
            return None
    else:
        if hoption == 3:
            hc = _candidates(h0, 16)
            ll = _loglik(x, y, wt, hc, m, cx, cy, case["cs"], dist, bud)
            if ll is None:
                return None
            h0 = hc[int(np.argmax(ll))]
        h = torch.full_like(x, float(h0))
    ew, pairs = _ec(x, y, h, m, cx, cy, case["cs"], dist, bud)
    if ew is None:
        return None
    den = _cells(x, y, _coef(wt, ew, _h2(h)), _h2(h), cx, cy, bud)
    if den is None:
        return None
    return {"density": _raster(den, m), "h": h.double().cpu().numpy(), "ew": ew.cpu().numpy(), "pairs": pairs,
            "h0": float(h0)}


def _loglik(x, y, w, hs, mask, cx, cy, cs, dist, bud):
    out = []
    for h in hs:
        hh = torch.full_like(x, float(h))
        ew, _ = _ec(x, y, hh, mask, cx, cy, cs, dist, bud)
        den = None if ew is None else _point_density(x, y, _coef(w, ew, _h2(hh)), _h2(hh), True, bud)
        if den is None:
            return None
        out.append(float(torch.log(den.clamp(min=EPS_DEN)).sum()))
    return np.array(out)


def exact(case, seed):
    kind = case["kind"]
    bud = _Budget()
    if kind == "ingest":
        return None            # copies and comparisons of inputs: nothing is rounded
    if kind == "serve":
        out = []
        for j, x, y, m in _serve_jobs(case, seed):
            e = _exact_job(j, x, y, None, m, j["hoption"], bud)
            if e is None:
                return None
            out.append((e["density"], None))
        return out
    if kind in ("job", "points", "search", "adaptive") and _too_large(case):
        return None
    x, y, w = _points(case, seed)
    if kind == "job":
        e = _exact_job(case, x, y, w, _mask(case, seed), case["hoption"], bud)
        return None if e is None else {k: e[k] for k in ("density", "h", "ew")}
    h0 = _rule(x, y, w)
    hs = _bandwidths(case, x, y, w, seed) if kind == "tile" else None
    wt = _t(np.ones(len(x), np.float32) if w is None else w)
    x, y = _t(x), _t(y)
    if kind == "raster":
        h = torch.full_like(x, float(np.float32(case["h"])))
        out = np.zeros((case["nrows"], case["ncols"]))
        top = _extent(case)
        for r in range(0, case["nrows"], case["tile"]):
            for c in range(0, case["ncols"], case["tile"]):
                nr, nc = min(case["tile"], case["nrows"] - r), min(case["tile"], case["ncols"] - c)
                cx, cy = _centres(nc, nr, np.float32(c * case["cs"]), np.float32(top - (r + nr) * case["cs"]),
                                  case["cs"])
                den = _cells(x, y, _coef(wt, 1.0, _h2(h)), _h2(h), _t(cx), _t(cy), bud)
                if den is None:
                    return None
                out[r:r + nr, c:c + nc] = den.cpu().numpy()
        return out
    if kind == "tile":
        h = _t(hs) if case["per_point"] else torch.full_like(x, float(hs))
        cx, cy = (_t(v) for v in _centres(case["ncols"], case["nrows"], 0.0, 0.0, np.float32(case["cs"])))
        if case["ec_cells"]:
            k = case["ec_cells"]
            ecs = float(np.float32(_extent(case) / k))
            ex, ey = (_t(v) for v in _centres(k, k, 0.0, 0.0, ecs))
            m, tm = torch.ones((k, k), device=_dev()), None
        else:
            ex, ey, ecs = cx, cy, float(case["cs"])
            m = tm = _t(_mask(case, seed))
        ew, _ = _ec(x, y, h, m, ex, ey, ecs, _boundary_dist(x, y, m, ex, ey), bud)
        den = None if ew is None else _cells(x, y, _coef(wt, ew, _h2(h)), _h2(h), cx, cy, bud)
        return None if den is None else {"ew": ew.cpu().numpy(), "density": _raster(den, tm)}
    m = _t(_mask(case, seed))
    cs = float(case["cs"])
    cx, cy = (_t(v) for v in _centres(case["ncols"], case["nrows"], 0.0, 0.0, cs))
    dist = _boundary_dist(x, y, m, cx, cy)
    if kind == "search":
        return _loglik(x, y, wt, _candidates(h0, case["k"], case["lo"], case["hi"]), m, cx, cy, cs, dist, bud)
    pairs = [(float(h0), -0.5)] if kind == "points" else list(zip(*(v.tolist() for v in _pairs(case, float(h0)))))
    lls = []
    for hp, alpha in pairs:
        den0, h = _adapt(x, y, wt, np.float32(hp), alpha, m, cx, cy, cs, dist, bud)
        ew = None if h is None else _ec(x, y, h, m, cx, cy, cs, dist, bud)[0]
        den1 = None if ew is None else _point_density(x, y, _coef(wt, ew, _h2(h)), _h2(h), True, bud)
        if den1 is None:
            return None
        if kind == "points":
            return {"h": h.double().cpu().numpy(), "den0": den0.cpu().numpy(), "ew": ew.cpu().numpy(),
                    "den1": den1.cpu().numpy()}
        lls.append(float(torch.log(den1.clamp(min=EPS_DEN)).sum()))
    return np.array(lls)


def _too_large(case):
    """Whether the pairs of the whole case are plainly beyond EXACT_PAIRS."""
    n, k = float(case["n"]), case.get("k", 1)
    if case["kind"] == "search":
        h = _candidates(_typical_h(case, case["n"]), k, case["lo"], case["hi"]).astype(float)
        wide = min(case["ncols"], case["nrows"])
        cells = np.minimum(6.0 * h / case["cs"], wide) ** 2
        share = np.minimum(1.0, math.pi * (3.0 * h) ** 2 / (case["ncols"] * case["nrows"] * case["cs"] ** 2))
        return bool((0.5 * n * cells + 2.0 * n * n * share).sum() > EXACT_PAIRS)
    cells = (6.0 * _typical_h(case, case["n"]) / case["cs"]) ** 2
    return 0.2 * n * cells * k > EXACT_PAIRS or (case["kind"] == "job" and 2.0 * n * cells > EXACT_PAIRS)
