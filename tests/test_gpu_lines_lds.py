"""Count lines drawn through LDS boxes (axis 0: runs of segments; axis 1 with a shared x:
strips) at the sizes and shapes where a box or a walk can go wrong, against the oracle.
Counts are whole numbers: bit-exact."""
from __future__ import annotations

import numpy as np
import pandas as pd
import pytest

import oracle

import golden_utils as G

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import datashader_amd as dsa  # noqa: E402


def _vertices(shape, n, rng):
    if shape == "series":
        return np.arange(n, dtype=np.float64), np.cumsum(rng.normal(0, 1, n)) + rng.normal(0, 20, n)
    x, y = np.cumsum(rng.normal(0, 1, (2, n)), axis=1)
    if shape == "jumps":       # every segment crosses the canvas: bounds beyond any box
        return rng.uniform(0, 1, n), rng.uniform(0, 1, n)
    if shape == "hops":        # the track jumps now and then: the box moves
        x = x + 1e3 * rng.integers(0, 9, n // 5000 + 1).repeat(5000)[:n]
    if shape == "gaps":
        x[rng.random(n) < 0.01] = np.nan
        y[rng.random(n) < 0.01] = np.nan
    if shape == "still":       # one place, then one long way back and forth
        x, y = np.zeros(n), np.zeros(n)
        x[n // 2], y[n // 2 + 1] = 1.0, 1.0
    return x, y


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [16384, 16385, 70001])
@pytest.mark.parametrize("shape,W,H,zoom", [
    ("series", 900, 525, False), ("track", 1901, 1080, False), ("jumps", 700, 300, False),
    ("hops", 640, 480, False), ("gaps", 333, 217, True), ("still", 1200, 900, False),
    ("series", 50_000, 3, False), ("track", 3, 50_000, True)])
def test_axis0_runs_vs_oracle(shape, W, H, zoom, n, dtype):
    x, y = _vertices(shape, n, np.random.default_rng(n))
    x, y = x.astype(dtype), y.astype(dtype)
    lo = [float(np.nanmin(v)) for v in (x, y)]
    hi = [float(np.nanmax(v)) for v in (x, y)]
    if zoom:  # a view with the data all around it
        lo, hi = [a + (b - a) / 4 for a, b in zip(lo, hi)], [b - (b - a) / 4 for a, b in zip(lo, hi)]
    xr, yr = (lo[0], hi[0]), (lo[1], hi[1])
    frame = dsa.DeviceFrame({"x": torch.as_tensor(x, device="cuda"),
                             "y": torch.as_tensor(y, device="cuda")})
    got = dsa.Canvas(W, H, x_range=xr, y_range=yr).line(frame, "x", "y", agg=dsa.count()).values
    f32 = dtype == np.float32
    view = G.view_for(W, H, xr, yr, xf32=f32, yf32=f32)
    exp = oracle.line_axis0(x.astype(np.float64), y.astype(np.float64), view, W, H)["count"]
    np.testing.assert_array_equal(got, exp)


def test_axis0_several_lines_and_strides_vs_oracle():
    rng = np.random.default_rng(3)
    n, m, W, H = 9001, 3, 400, 300
    xs, ys = np.cumsum(rng.normal(0, 1, (2, n, m)), axis=1)
    tx, ty = torch.as_tensor(xs, device="cuda"), torch.as_tensor(ys, device="cuda")
    cols = {f"x{j}": tx[:, j] for j in range(m)} | {f"y{j}": ty[:, j] for j in range(m)}
    agg = dsa.Canvas(W, H).line(dsa.DeviceFrame(cols), x=[f"x{j}" for j in range(m)],
                                y=[f"y{j}" for j in range(m)], agg=dsa.count())
    view = G.view_for(W, H, agg.x_range, agg.y_range)
    exp = sum(oracle.line_axis0(xs[:, j].copy(), ys[:, j].copy(), view, W, H)["count"].astype(int)
              for j in range(m))
    np.testing.assert_array_equal(agg.values, exp)


@pytest.mark.parametrize("axis_type", ["linear", "log"])
@pytest.mark.parametrize("nverts,W,H", [
    (5, 2000, 300),     # 400 columns a segment: walks beyond the fixed-point steps
    (33, 300, 1080), (256, 700, 90), (300, 1900, 1080)])
@pytest.mark.parametrize("ydtype", [np.float32, np.float64])
def test_shared_x_strips_vs_oracle(nverts, W, H, ydtype, axis_type):
    rng = np.random.default_rng(nverts)
    nlines = 1025
    xs = np.linspace(1.0, 9.0, nverts)
    if nverts == 33:
        xs = xs[::-1].copy()
    ys = (5 + np.cumsum(rng.normal(0, 0.4, (nlines, nverts)), axis=1)).astype(ydtype)
    ys[rng.random(ys.shape) < 0.01] = np.nan
    xr, yr = (1.0, 9.0), (2.0, 8.0)
    names = [f"y{j}" for j in range(nverts)]
    frame = dsa.DeviceFrame.from_pandas(pd.DataFrame(ys, columns=names))
    cvs = dsa.Canvas(W, H, x_range=xr, y_range=yr, x_axis_type="linear", y_axis_type=axis_type)
    got = cvs.line(frame, x=xs, y=names, agg=dsa.count(), axis=1).values
    if axis_type == "log":  # the oracle has linear axes: the general kernel is the reference
        X = torch.as_tensor(np.tile(xs, (nlines, 1)), device="cuda")
        cols = {n: frame[n] for n in names} | {f"x{j}": X[:, j] for j in range(nverts)}
        exp = cvs.line(dsa.DeviceFrame(cols), x=[f"x{j}" for j in range(nverts)], y=names,
                       agg=dsa.count(), axis=1).values
    else:
        view = G.view_for(W, H, xr, yr, yf32=ydtype == np.float32)
        exp = oracle.lines_xconst(xs, ys.astype(np.float64), view, W, H)["count"]
    assert exp.sum() > 0
    np.testing.assert_array_equal(got, exp)
