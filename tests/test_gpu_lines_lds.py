"""Count lines drawn through LDS boxes (axis 1 with a shared x: strips) at the sizes and shapes where a box or a walk can go wrong, against the oracle.
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
