"""How axis-0 count lines are shared out over workgroups, against the oracle: lines split into
several runs, runs of many rounds (the box held, moved, kept though the pixels leave it, rounds
with nothing to draw).  Counts are whole numbers: bit-exact."""
from __future__ import annotations

import numpy as np
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


@pytest.mark.parametrize("m,n", [(3, 9001), (257, 4097), (300, 6145), (520, 4099)])
def test_lines_split_into_runs(m, n):
    rng = np.random.default_rng(m)
    xs, ys = np.cumsum(rng.normal(0, 1, (2, m, n)), axis=2).astype(np.float32)
    got, exp = _lines(xs, ys, 640, 360, (-120.0, 120.0), (-90.0, 90.0))
    assert exp.sum() > 0
    np.testing.assert_array_equal(got, exp)
