"""The work the performance of this package is measured on.

Each case is one call that a user's program makes through the public entry points
(``Canvas.points``, ``Canvas.line``, ``tf.shade``, ``BatchServer.serve``), on inputs made
from a seed.  ``listed()`` names the fixed cases, ``draw(rng)`` gives further ones of the
same ranges, ``prepare`` makes what the program has in hand before the call, ``run`` makes
the call, ``work`` states the bytes it cannot do without, and ``exact`` recomputes the
floating-point outputs in 64 bits with plain torch.
"""
import math

import numpy as np
import torch

import datashader_amd as dsa
import datashader_amd.transfer_functions as tf
from datashader_amd import batching, serving

DEVICE = "cuda"


def listed():
    return [
        # an interactive view of a small table: launches and host time count
        dict(name="points_small", kind="points", rows=100_000, width=600, height=600,
             spread="mixture", dtype="f32", agg="count", ncat=0, autorange=False),
        # an ordinary scatter plot of a double-precision table with missing rows
        dict(name="points_800x600_f64", kind="points", rows=10_000_000, width=800, height=600,
             spread="mixture", dtype="f64", agg="count", ncat=0, autorange=False),
        # the headline: a large table, most of it in one hot spot, on a full HD canvas
        dict(name="points_skewed_100m", kind="points", rows=100_000_000, width=1920, height=1080,
             spread="cluster", dtype="f32", agg="count_mean", ncat=0, autorange=False),
        # the largest table, coloured by category
        dict(name="points_bycat_500m", kind="points", rows=500_000_000, width=1024, height=1024,
             spread="ridges", dtype="f32", agg="by_count", ncat=16, autorange=False),
        # a statistics panel (count, sum, min, max, std) over a table spread over the whole
        # canvas, ranges taken from the data, odd sizes
        dict(name="points_stats_f64", kind="points", rows=20_000_003, width=1023, height=767,
             spread="uniform", dtype="f64", agg="stats", ncat=0, autorange=True),
        # the mean of a value per category
        dict(name="points_bymean", kind="points", rows=50_000_000, width=700, height=500,
             spread="mixture", dtype="f32", agg="by_mean", ncat=8, autorange=False),
        # hover information: a column of the row with the largest value of each pixel
        dict(name="points_where_max", kind="points", rows=50_000_001, width=1200, height=900,
             spread="cluster", dtype="f32", agg="where_max", ncat=0, autorange=False),
        # many sampled series on one time axis
        dict(name="lines_shared_x", kind="lines", rows=1_000_000, samples=256, width=2048,
             height=1024, dtype="f32", agg="count", autorange=False),
        # one long time series
        dict(name="line_series", kind="series", rows=10_000_000, width=900, height=525,
             shape="time", dtype="f64", agg="any", autorange=True),
        # colouring a full HD aggregate by histogram equalisation
        dict(name="shade_eq_hist", kind="shade", rows=20_000_000, width=1920, height=1080,
             spread="cluster", plane="count", ncat=0, how="eq_hist"),
        # a batch of map viewports over a resident table
        dict(name="served_viewports", kind="served", rows=100_000_000, requests=24, grid=1024),
        # a pandas table from host memory to a host result, ranges taken from the data
        dict(name="points_pandas", kind="pandas", rows=3_000_000, width=900, height=600,
             spread="mixture", dtype="f64", agg="count_mean", autorange=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["points", "points", "points", "points", "bycat", "bycat", "select",
                       "lines", "series", "shade", "served", "pandas"])
    w, h = rng.randint(200, 1920), rng.randint(150, 1080)
    dtype = rng.choice(["f32", "f32", "f64"])
    spread = rng.choice(["mixture", "cluster", "uniform", "ridges"])
    auto = rng.random() < 0.4
    if kind == "points":
        return dict(kind="points", rows=_log_int(rng, 10_000, 100_000_000), width=w, height=h,
                    spread=spread, dtype=dtype, ncat=0, autorange=auto,
                    agg=rng.choice(["count", "count_mean", "mean", "stats"]))
    if kind == "bycat":
        return dict(kind="points", rows=_log_int(rng, 100_000, 100_000_000),
                    width=rng.randint(200, 1024), height=rng.randint(150, 1024), spread=spread,
                    dtype=dtype, ncat=rng.randint(2, 16), autorange=auto,
                    agg=rng.choice(["by_count", "by_mean"]))
    if kind == "select":
        return dict(kind="points", rows=_log_int(rng, 100_000, 50_000_000), width=w, height=h,
                    spread=spread, dtype="f32", ncat=0, autorange=auto,
                    agg=rng.choice(["first", "last", "where_max", "where_min", "max_n"]))
    if kind == "lines":
        samples = rng.randint(32, 300)
        return dict(kind="lines", rows=_log_int(rng, 1_000, 200_000_000 // samples),
                    samples=samples, width=rng.randint(300, 2048), height=rng.randint(200, 1080),
                    dtype=dtype, agg=rng.choice(["count", "any"]), autorange=auto)
    if kind == "series":
        return dict(kind="series", rows=_log_int(rng, 10_000, 10_000_000), width=w, height=h,
                    shape=rng.choice(["time", "track"]), dtype=dtype,
                    agg=rng.choice(["any", "count"]), autorange=auto)
    if kind == "shade":
        plane = rng.choice(["count", "mean", "cat"])
        return dict(kind="shade", rows=_log_int(rng, 100_000, 20_000_000), width=w, height=h,
                    spread=spread, plane=plane, ncat=rng.randint(2, 16) if plane == "cat" else 0,
                    how=rng.choice(["eq_hist", "eq_hist", "log", "linear"]))
    if kind == "served":
        return dict(kind="served", rows=_log_int(rng, 1_000_000, 100_000_000),
                    requests=rng.randint(4, 24), grid=1024)
    return dict(kind="pandas", rows=_log_int(rng, 10_000, 3_000_000), width=w, height=h,
                spread=spread, dtype=dtype, agg=rng.choice(["count", "count_mean"]),
                autorange=auto)


# ---- inputs ---------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _xy(spread, n, g, dtype):
    """n points in or near the unit square."""
    def rand():
        return torch.rand(n, generator=g, device=DEVICE, dtype=dtype)

    def randn():
        return torch.randn(n, generator=g, device=DEVICE, dtype=dtype)

    if spread == "uniform":
        return rand(), rand()
    if spread == "cluster":  # 90 % in a narrow Gaussian, 10 % everywhere, in random order
        hot = torch.rand(n, generator=g, device=DEVICE) < 0.9
        x, y = rand(), rand()
        zx, zy = randn(), randn()
        x = torch.where(hot, zx.mul_(0.01).add_(0.5), x)
        del zx
        return x, torch.where(hot, zy.mul_(0.01).add_(0.5), y)
    if spread == "ridges":  # 40 % uniform, 60 % along three curves
        x, y = rand(), rand()
        k = torch.randint(1, 4, (n,), generator=g, device=DEVICE, dtype=torch.int32).to(dtype)
        r = (x * k).mul_(2 * math.pi).sin_().mul_(0.1).add_(k, alpha=0.25)
        del k
        r += randn().mul_(0.02)
        on = torch.rand(n, generator=g, device=DEVICE) < 0.6
        return x, torch.where(on & (r >= 0) & (r <= 1), r, y)
    # five Gaussians, one row in a thousand missing
    means = torch.rand(2, 5, generator=g, device=DEVICE, dtype=dtype) * 0.6 + 0.2
    sigma = torch.rand(5, generator=g, device=DEVICE, dtype=dtype) * 0.065 + 0.01
    comp = torch.randint(0, 5, (n,), generator=g, device=DEVICE)
    x = randn().mul_(sigma[comp]).add_(means[0][comp])
    y = randn().mul_(sigma[comp]).add_(means[1][comp])
    miss = torch.randint(0, n, (max(1, n // 1000),), generator=g, device=DEVICE)
    x[miss] = float("nan")
    y[miss] = float("nan")
    return x, y


def _columns(case, seed):
    g = _gen(seed)
    n = case["rows"]
    dt = torch.float64 if case["dtype"] == "f64" else torch.float32
    x, y = _xy(case["spread"], n, g, dt)
    cols = {"x": x, "y": y}
    agg = case["agg"]
    if agg in ("count_mean", "mean", "stats", "by_mean", "first", "last", "where_max",
               "where_min", "max_n"):
        v = torch.randn(n, generator=g, device=DEVICE, dtype=dt).mul_(1.5).exp_()
        if agg in ("mean", "stats", "first", "last"):  # a few missing values
            v[torch.randint(0, n, (max(1, n // 500),), generator=g, device=DEVICE)] = float("nan")
        cols["v"] = v
    if agg in ("where_max", "where_min"):
        cols["w"] = torch.rand(n, generator=g, device=DEVICE)
    if agg in ("by_count", "by_mean"):  # Zipf(1.2) categories
        p = np.arange(1, case["ncat"] + 1, dtype=np.float64) ** -1.2
        cdf = torch.tensor(np.cumsum(p / p.sum()), dtype=torch.float32, device=DEVICE)
        code = torch.empty(n, dtype=torch.int8, device=DEVICE)
        for s in range(0, n, 1 << 26):
            m = min(1 << 26, n - s)
            u = torch.rand(m, generator=g, device=DEVICE)
            code[s:s + m] = torch.searchsorted(cdf, u).clamp_(max=case["ncat"] - 1).to(torch.int8)
        cols["cat"] = code
    return cols


def _reduction(agg):
    return {
        "count": lambda: dsa.count(),
        "any": lambda: dsa.any(),
        "mean": lambda: dsa.mean("v"),
        "count_mean": lambda: dsa.summary(count=dsa.count(), mean=dsa.mean("v")),
        "stats": lambda: dsa.summary(n=dsa.count("v"), total=dsa.sum("v"), low=dsa.min("v"),
                                     high=dsa.max("v"), std=dsa.std("v")),
        "by_count": lambda: dsa.by("cat", dsa.count()),
        "by_mean": lambda: dsa.by("cat", dsa.mean("v")),
        "first": lambda: dsa.first("v"),
        "last": lambda: dsa.last("v"),
        "where_max": lambda: dsa.where(dsa.max("v"), "w"),
        "where_min": lambda: dsa.where(dsa.min("v"), "w"),
        "max_n": lambda: dsa.max_n("v", n=3),
    }[agg]()


# the view of a call that gives its ranges: most of the unit square, a margin left out
VIEW = ((0.02, 0.98), (0.03, 0.97))


def _canvas(case):
    if case["autorange"]:
        return dsa.Canvas(case["width"], case["height"])
    return dsa.Canvas(case["width"], case["height"], x_range=VIEW[0], y_range=VIEW[1])


def _frame(case, cols):
    cats = {"cat": ["c%d" % k for k in range(case["ncat"])]} if "cat" in cols else None
    return dsa.DeviceFrame(cols, categories=cats)


def _walks(case, seed):
    """[samples, series] random walks from -1 .. 1, and their shared sample times."""
    g = _gen(seed)
    m, n = case["samples"], case["rows"]
    dt = torch.float64 if case["dtype"] == "f64" else torch.float32
    block = torch.empty(m, n, dtype=dt, device=DEVICE)
    block[0] = torch.rand(n, generator=g, device=DEVICE, dtype=dt) * 2 - 1
    for j in range(1, m):
        torch.randn(n, generator=g, device=DEVICE, dtype=dt, out=block[j])
        block[j].mul_(0.02).add_(block[j - 1])
    return np.linspace(0.0, 1.0, m), block


def _series(case, seed):
    g = _gen(seed)
    n = case["rows"]
    dt = torch.float64 if case["dtype"] == "f64" else torch.float32

    def walk(step):
        return torch.randn(n, generator=g, device=DEVICE, dtype=torch.float64).mul_(step).cumsum(0)

    if case["shape"] == "time":  # evenly sampled time, a slow walk under measurement noise
        x = torch.arange(n, device=DEVICE, dtype=torch.float64)
        y = walk(1.0 / math.sqrt(n)) + 0.02 * torch.randn(n, generator=g, device=DEVICE,
                                                          dtype=torch.float64)
    else:  # a track over the plane, with some fixes missing
        x, y = walk(1.0 / math.sqrt(n)), walk(1.0 / math.sqrt(n))
        miss = torch.randint(0, n, (max(1, n // 1000),), generator=g, device=DEVICE)
        x[miss] = float("nan")
    return x.to(dt), y.to(dt)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "points":
        return dict(call="points", canvas=_canvas(case), frame=_frame(case, _columns(case, seed)),
                    agg=_reduction(case["agg"]))
    if kind == "pandas":
        import pandas as pd
        cols = {k: c.cpu().numpy() for k, c in _columns(case, seed).items()}
        return dict(call="points", canvas=_canvas(case), frame=pd.DataFrame(cols),
                    agg=_reduction(case["agg"]))
    if kind == "lines":
        xs, block = _walks(case, seed)
        names = ["y%d" % j for j in range(case["samples"])]
        if case["autorange"]:
            cvs = dsa.Canvas(case["width"], case["height"])
        else:
            cvs = dsa.Canvas(case["width"], case["height"], x_range=(0.0, 1.0),
                             y_range=(-2.0, 2.0))
        return dict(call="lines", canvas=cvs, frame=dsa.DeviceFrame.from_block(names, block),
                    x=xs, y=names, agg=_reduction(case["agg"]))
    if kind == "series":
        x, y = _series(case, seed)
        if case["autorange"]:
            cvs = dsa.Canvas(case["width"], case["height"])
        else:  # a view of the middle half of the data
            x0, x1, y0, y1 = (float(t) for t in (x.nan_to_num(0.0).min(), x.nan_to_num(0.0).max(),
                                                 y.min(), y.max()))
            cvs = dsa.Canvas(case["width"], case["height"],
                             x_range=(x0 + (x1 - x0) / 4, x1 - (x1 - x0) / 4),
                             y_range=(y0 + (y1 - y0) / 4, y1 - (y1 - y0) / 4))
        return dict(call="lines", canvas=cvs, frame=dsa.DeviceFrame({"x": x, "y": y}), x="x",
                    y="y", agg=_reduction(case["agg"]))
    if kind == "shade":
        agg = {"count": "count", "mean": "mean", "cat": "by_count"}[case["plane"]]
        full = dict(case, agg=agg, dtype="f32", autorange=False)
        frame = _frame(full, _columns(full, seed))
        return dict(call="shade", plane=_canvas(full).points(frame, "x", "y", _reduction(agg)),
                    how=case["how"])
    # served: a resident table, its index and server, and a page of requests
    g = _gen(seed)
    x, y = _xy("mixture", case["rows"], g, torch.float32)
    x, y = x.nan_to_num_(0.5), y.nan_to_num_(0.5)
    v = torch.rand(case["rows"], generator=g, device=DEVICE)
    index = serving.PointIndex(x, y, v, grid=case["grid"])
    server = batching.BatchServer(index, engines=2, max_batch=32)
    return dict(call="served", server=server, requests=_requests(case, seed, x, y))


def _sizes(case):
    return [((1920, 1080), (256, 256), (1024, 768), (512, 512))[k % 4]
            for k in range(case["requests"])]


def _requests(case, seed, x, y):
    """Viewports centred on rows of the table, zoomed in by up to 2^10."""
    rng = np.random.default_rng(seed)
    at = torch.from_numpy(rng.integers(0, case["rows"], case["requests"])).to(DEVICE)
    cx, cy = x[at].cpu().numpy(), y[at].cpu().numpy()
    out = []
    for k, (w, h) in enumerate(_sizes(case)):
        half = 0.5 * 2.0 ** -rng.uniform(0, 10)
        out.append(serving.Request((float(cx[k]) - half, float(cx[k]) + half),
                                   (float(cy[k]) - half, float(cy[k]) + half), w, h,
                                   dsa.summary(count=dsa.count(), mean=dsa.mean("v"))))
    return out


# ---- the calls ------------------------------------------------------------------------

def _plane(a):
    """The array of a result; device counts and pixels (torch.uint32) as int32 bits."""
    a = a.data
    if isinstance(a, torch.Tensor) and a.dtype == torch.uint32:
        return a.view(torch.int32)
    return a


def _outputs(res, keys):
    return _plane(res) if keys is None else {k: _plane(res[k]) for k in keys}


def _keys(agg):
    return list(agg.keys) if isinstance(agg, dsa.summary) else None


def run(state):
    call = state["call"]
    if call == "points":
        res = state["canvas"].points(state["frame"], "x", "y", state["agg"])
        return _outputs(res, _keys(state["agg"]))
    if call == "lines":
        res = state["canvas"].line(state["frame"], x=state["x"], y=state["y"], agg=state["agg"],
                                   axis=0 if state["x"] is not None and isinstance(state["x"], str)
                                   else 1)
        return _outputs(res, None)
    if call == "shade":
        return _plane(tf.shade(state["plane"], how=state["how"]))
    done = state["server"].serve(state["requests"], realtime=False, keep_results=True)
    return [_outputs(r, ("count", "mean")) for r in done["results"]]


def work(case):
    """Bytes of each input read once and each output written once."""
    kind, n = case["kind"], case["rows"]
    cells = case.get("width", 0) * case.get("height", 0)
    item = 8 if case.get("dtype") == "f64" else 4
    if kind in ("points", "pandas"):
        agg = case["agg"]
        cols = 2 + (agg not in ("count", "by_count"))
        nbytes = cols * item * n
        out = {"count": 4, "mean": 8, "count_mean": 12, "stats": 4 + 4 * 8,
               "by_count": 4 * case.get("ncat", 0), "by_mean": 8 * case.get("ncat", 0),
               "max_n": 24}.get(agg, 8)
        if agg.startswith("by_"):
            nbytes += n
        if agg.startswith("where"):  # one looked-up value a cell at most
            nbytes += 4 * min(n, cells)
        return {"bytes": nbytes + out * cells, "flops": 0}
    out = 1 if case.get("agg") == "any" else 4
    if kind == "lines":
        return {"bytes": item * n * case["samples"] + 8 * case["samples"] + out * cells, "flops": 0}
    if kind == "series":
        return {"bytes": 2 * item * n + out * cells, "flops": 0}
    if kind == "shade":
        plane = {"count": 4, "mean": 8, "cat": 4 * case["ncat"]}[case["plane"]]
        return {"bytes": (plane + 4) * cells, "flops": 0}
    # the table once, and every request's two planes
    return {"bytes": 12 * n + 12 * sum(w * h for w, h in _sizes(case)), "flops": 0}


# ---- 64-bit recomputation of the floating-point outputs ---------------------------------

def _bins(x, y, xr, yr, w, h, cat=None, ncat=1):
    """Cell of each row (the float64 projection, truncated; the upper edge into the last
    bin); -1 for rows outside the view."""
    x, y = x.double(), y.double()
    keep = (x >= xr[0]) & (x <= xr[1]) & (y >= yr[0]) & (y <= yr[1])

    def pixel(v, r, m):
        s = m / (r[1] - r[0])
        return (v.nan_to_num(r[0]).clamp(r[0], r[1]) * s + (-r[0] * s)).long().clamp(max=m - 1)

    cell = pixel(y, yr, h) * w + pixel(x, xr, w)
    if cat is not None:
        cell = cell * ncat + cat.long()
    return torch.where(keep, cell, -1)


def _rows_of(x, y, xr, yr, w, h, cat=None, ncat=1):
    """(cells, row numbers) of the rows inside the view, in blocks of 2^25 rows."""
    cells, rows = [], []
    for s in range(0, x.shape[0], 1 << 25):
        e = s + (1 << 25)
        c = _bins(x[s:e], y[s:e], xr, yr, w, h, None if cat is None else cat[s:e], ncat)
        r = torch.nonzero(c >= 0).flatten()
        cells.append(c[r])
        rows.append(r + s)
    return torch.cat(cells), torch.cat(rows)


def _per_cell(cell, v, size):
    """(values, sum) per cell of the rows with a value."""
    ok = ~torch.isnan(v)
    c, v = cell[ok], v[ok].double()
    n = torch.zeros(size, dtype=torch.float64, device=DEVICE).index_add_(0, c, torch.ones_like(v))
    return c, v, n, torch.zeros(size, dtype=torch.float64, device=DEVICE).index_add_(0, c, v)


def _nan_where(empty, a):
    return torch.where(empty, torch.full_like(a, float("nan")), a)


def _exact_points(case, cols, xr, yr):
    agg = case["agg"]
    if agg in ("count", "by_count"):
        return None
    w, h = case["width"], case["height"]
    ncat = case.get("ncat") or 1
    shape = (h, w, ncat) if agg.startswith("by_") else (h, w)
    size = h * w * ncat
    cell, rows = _rows_of(cols["x"], cols["y"], xr, yr, w, h, cols.get("cat"), ncat)
    v = cols["v"][rows]
    if agg in ("mean", "count_mean", "by_mean", "stats"):
        c, vv, n, total = _per_cell(cell, v, size)
        mean = total / n
        if agg in ("mean", "by_mean"):
            return mean.reshape(shape)
        if agg == "count_mean":
            return {"count": None, "mean": mean.reshape(shape)}
        m2 = torch.zeros_like(total).index_add_(0, c, (vv - mean[c]) ** 2)
        inf = torch.full_like(total, float("inf"))
        low = inf.clone().scatter_reduce_(0, c, vv, "amin")
        high = (-inf).scatter_reduce_(0, c, vv, "amax")
        none = n == 0
        return {"n": None, "total": _nan_where(none, total).reshape(shape),
                "low": _nan_where(none, low).reshape(shape),
                "high": _nan_where(none, high).reshape(shape),
                "std": torch.sqrt(m2 / n).reshape(shape)}
    # selections of rows: the first or last with a value, or the first of the extreme value
    ok = ~torch.isnan(v)
    cell, rows, v = cell[ok], rows[ok], v[ok].double()
    if agg == "max_n":
        left = torch.ones_like(v, dtype=torch.bool)
        out = []
        for _ in range(3):
            row = _first_extreme(cell[left], rows[left], v[left], size, "amax")
            out.append(_take(row, cols["v"]))
            taken = torch.zeros(cols["v"].shape[0], dtype=torch.bool, device=DEVICE)
            taken[row[row < _FAR]] = True
            left &= ~taken[rows]
        return torch.stack(out, -1).reshape(h, w, 3)
    if agg in ("first", "last"):
        empty = _FAR if agg == "first" else -1
        row = torch.full((size,), empty, dtype=torch.int64, device=DEVICE)
        row.scatter_reduce_(0, cell, rows, "amin" if agg == "first" else "amax")
        row = torch.where(row < 0, _FAR, row)
        return _take(row, cols["v"]).reshape(shape)
    row = _first_extreme(cell, rows, v, size, "amax" if agg == "where_max" else "amin")
    return _take(row, cols["w"]).reshape(shape)


_FAR = 1 << 40  # no row


def _first_extreme(cell, rows, v, size, how):
    """First row of each cell that has the cell's extreme value."""
    best = torch.full((size,), -math.inf if how == "amax" else math.inf, dtype=torch.float64,
                      device=DEVICE).scatter_reduce_(0, cell, v, how)
    at = v == best[cell]
    return torch.full((size,), _FAR, dtype=torch.int64,
                      device=DEVICE).scatter_reduce_(0, cell[at], rows[at], "amin")


def _take(row, col):
    none = row >= _FAR
    return _nan_where(none, col.double()[torch.where(none, 0, row)])


def _range_of(col):
    ok = col[~torch.isnan(col)]
    return float(ok.min()), float(ok.max())


def exact(case, seed):
    if case["kind"] in ("points", "pandas"):
        if case["agg"] in ("count", "by_count"):
            return None
        cols = _columns(case, seed)
        xr, yr = VIEW
        if case["autorange"]:
            xr, yr = _range_of(cols["x"]), _range_of(cols["y"])
        return _exact_points(case, cols, xr, yr)
    if case["kind"] != "served":
        return None  # pixels: whole numbers
    g = _gen(seed)
    x, y = _xy("mixture", case["rows"], g, torch.float32)
    x, y = x.nan_to_num_(0.5), y.nan_to_num_(0.5)
    v = torch.rand(case["rows"], generator=g, device=DEVICE)
    out = []
    for r in _requests(case, seed, x, y):
        cell, rows = _rows_of(x, y, r.x_range, r.y_range, r.width, r.height)
        _, _, n, total = _per_cell(cell, v[rows], r.width * r.height)
        out.append({"count": None, "mean": (total / n).reshape(r.height, r.width)})
    return out
