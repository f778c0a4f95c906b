"""How axis-0 count lines are shared out over workgroups, against the oracle: lines split into
several runs, runs of many rounds (the box held, moved, kept though the pixels leave it, rounds
with nothing to draw).  Counts are whole numbers: bit-exact."""
from __future__ import annotations

import numpy as np
import pandas as pd
import pytest

import oracle

import golden_utils as G

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import datashader_amd as dsa  # noqa: E402


def _lines(xs, ys, W, H, xr, yr):
    """Counts of the lines xs[j], ys[j] and the oracle's."""
    m = len(xs)
    tx, ty = torch.as_tensor(xs, device="cuda"), torch.as_tensor(ys, device="cuda")
    cols = {f"x{j}": tx[j] for j in range(m)} | {f"y{j}": ty[j] for j in range(m)}
    cvs = dsa.Canvas(W, H, x_range=xr, y_range=yr)
    got = cvs.line(dsa.DeviceFrame(cols), x=[f"x{j}" for j in range(m)],
                   y=[f"y{j}" for j in range(m)], agg=dsa.count()).values
    f32 = xs.dtype == np.float32
    view = G.view_for(W, H, xr, yr, xf32=f32, yf32=f32)
    exp = np.zeros((H, W), np.int64)
    for j in range(m):
        exp += oracle.line_axis0(xs[j].astype(np.float64), ys[j].astype(np.float64), view, W,
                                 H)["count"].astype(np.int64)
    return got, exp


@pytest.mark.parametrize("m,n", [(3, 10_924), (7, 9001), (257, 4097), (300, 6145), (520, 4099)])
def test_lines_split_into_runs(m, n):
    rng = np.random.default_rng(m)
    xs, ys = np.cumsum(rng.normal(0, 1, (2, m, n)), axis=2).astype(np.float32)
    got, exp = _lines(xs, ys, 640, 360, (-120.0, 120.0), (-90.0, 90.0))
    assert exp.sum() > 0
    np.testing.assert_array_equal(got, exp)


def _blocks(kind, n, rng):
    """A line whose stretches of 4096 vertices (a round of one workgroup) differ: near one place,
    near another, all over the view, all outside it, one vertex repeated, few in the view."""
    m = -(-n // 4096)
    x, y = np.cumsum(rng.normal(0, 0.02, (2, m, 4096)), axis=2)
    cx, cy = rng.uniform(5, 95, (2, m, 1))
    x, y = cx + x, cy + y
    what = rng.integers(0, 6, m) if kind == "mixed" else np.arange(m) % 2 * 3
    x[what == 2], y[what == 2] = rng.uniform(0, 100, (2, int((what == 2).sum()), 4096))
    x[what == 3] += 200  # (beyond the view)
    x[what == 4], y[what == 4] = cx[what == 4], cy[what == 4]
    out = (what == 5)[:, None] & (rng.random((m, 4096)) < 0.99)
    x[out] = np.nan
    return x.reshape(-1)[:n], y.reshape(-1)[:n]


@pytest.mark.parametrize("n", [32_768, 32_769, 32_770, 65_535])
@pytest.mark.parametrize("W,H", [(1900, 1000), (640, 1), (1, 480), (30_000, 4)])
def test_first_sizes(W, H, n):
    """The smallest lines drawn in runs (boxes no larger than a round's pixels), in full and with
    a view in the middle."""
    rng = np.random.default_rng(n)
    t = np.arange(n, dtype=np.float64)
    noisy = np.cumsum(rng.normal(0, 1, n)) + rng.normal(0, 9, n)
    track = np.cumsum(rng.normal(0, 1, (2, n)), axis=1)
    track[0][::97] = np.nan
    for x, y in ((t, noisy), (track[0], track[1])):
        for cut in (0.0, 0.25):
            xr, yr = ((float(np.nanquantile(a, cut)), float(np.nanquantile(a, 1 - cut))) for a in (x, y))
            got, exp = _lines(x[None], y[None], W, H, xr, yr)
            assert exp.sum() > 0
            np.testing.assert_array_equal(got, exp)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind,W,H", [("mixed", 300, 200), ("mixed", 90, 60), ("in_out", 700, 400),
                                      ("series", 300, 300), ("gaps", 640, 360)])
def test_many_rounds(kind, W, H, dtype):
    """One line of 13 thousand segments a workgroup, and 256 lines of one workgroup each."""
    rng = np.random.default_rng(W)
    for m, n in ((1, 3_300_001), (256, 12_901)):
        if kind in ("mixed", "in_out"):
            lines = [_blocks(kind, n, rng) for _ in range(m)]
            xr = yr = (0.0, 100.0)
        elif kind == "series":
            lines = [(np.arange(n) * (100.0 / n), 50 + rng.normal(0, 2, n)) for _ in range(m)]
            xr, yr = (0.0, 100.0), (40.0, 60.0)
        else:  # a track, fixes missing, most of it around the view
            lines = [tuple(np.cumsum(rng.normal(0, 0.1, (2, n)), axis=1)) for _ in range(m)]
            for x, y in lines:
                x[rng.random(n) < 0.01] = np.nan
                y[::4099] = np.nan
            xr = yr = (-20.0, 20.0)
        xs, ys = (np.stack([q[i] for q in lines]).astype(dtype) for i in (0, 1))
        got, exp = _lines(xs, ys, W, H, xr, yr)
        assert exp.sum() > 0
        np.testing.assert_array_equal(got, exp)


@pytest.mark.parametrize("xt,yt", [("log", "linear"), ("linear", "log"), ("log", "log"),
                                   ("linear", "linear")])
@pytest.mark.parametrize("xd,yd", [("float32", "float32"), ("float64", "float32"),
                                   ("float32", "float64"), ("float64", "float64")])
def test_axes_and_types(xd, yd, xt, yt):
    """Against the general kernel, which a count of a column takes."""
    n = 60_001
    rng = np.random.default_rng(n)
    x = 1 + np.arange(n) * 0.01 + rng.uniform(0, 0.01, n)
    y = np.exp(np.cumsum(rng.normal(0, 0.01, n)) + rng.normal(0, 0.2, n))
    y[::501] = np.nan
    y[7::777] *= -1  # (not on a log axis)
    x, y = x.astype(xd), y.astype(yd)
    f = dsa.DeviceFrame({"x": torch.from_numpy(x).cuda(), "y": torch.from_numpy(y).cuda(),
                         "one": torch.ones(n, device="cuda")})
    for xr, yr in (((1.0, 601.0), (0.2, 5.0)), ((30.0, 90.0), (0.9, 1.1))):
        cvs = dsa.Canvas(700, 400, x_range=xr, y_range=yr, x_axis_type=xt, y_axis_type=yt)
        got = cvs.line(f, "x", "y", agg=dsa.count()).values
        exp = cvs.line(f, "x", "y", agg=dsa.count("one")).values
        assert exp.sum() > 0
        np.testing.assert_array_equal(got, exp)


@pytest.mark.parametrize("chunk_rows", [32_766, 32_769, 50_001])
def test_streamed_chunks(chunk_rows):
    """A line in chunks long enough for the runs: the vertices before a chunk are context, and a
    partition's first chunk goes on from the last partition's row without drawing it again."""
    n = 160_003
    rng = np.random.default_rng(chunk_rows)
    x, y = np.cumsum(rng.normal(0, 0.05, (2, n)), axis=1)
    for at in range(0, n, chunk_rows):  # (gaps at, before and after the chunks' first rows)
        x[at + int(rng.integers(-3, 3))] = np.nan
    y[rng.random(n) < 0.02] = np.nan
    df = pd.DataFrame({"x": x, "y": y, "one": 1.0})
    W, H = 257, 193
    cvs = dsa.Canvas(W, H)
    resident = cvs.line(df, "x", "y", agg=dsa.count())
    xr, yr = resident.attrs["x_range"], resident.attrs["y_range"]
    view = G.view_for(W, H, xr, yr)
    np.testing.assert_array_equal(resident.values, oracle.line_axis0(x, y, view, W, H)["count"])
    streamed = cvs.line(dsa.ChunkedFrame(df, chunk_rows=chunk_rows), "x", "y", agg=dsa.count())
    np.testing.assert_array_equal(streamed.values, resident.values)
    cuts = [0, 70_000, 105_000, n]
    parts = [df.iloc[a:b] for a, b in zip(cuts[:-1], cuts[1:])]
    got = cvs.line(dsa.ChunkedFrame(parts, chunk_rows=chunk_rows), "x", "y", agg=dsa.count())
    want = np.zeros((H, W), np.int64)
    for i, p in enumerate(parts):
        rows = p if i == 0 else pd.concat([parts[i - 1].iloc[-1:], p])
        want += oracle.line_axis0(rows["x"].to_numpy(), rows["y"].to_numpy(), view, W, H,
                                  plot_start=(i == 0))["count"]
    np.testing.assert_array_equal(got.values, want)
