"""Series on a shared x whose neighbouring lanes walk short, long and clipped segments in one
pass over the LDS strip, against the oracle.  Counts are whole numbers: bit-exact."""
from __future__ import annotations

import numpy as np
import pytest

import oracle

import golden_utils as G

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import datashader_amd as dsa  # noqa: E402


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("values", ["noise", "spikes", "flat"])
@pytest.mark.parametrize("nverts,W,H", [
    (2, 700, 1000),     # one segment a line, wider than the fixed-point steps
    (17, 200, 255),     # no walk beyond them
    (17, 200, 257),     # a step or two beyond
    (9, 30, 8192),      # the band takes all of the LDS
    (32, 1812, 803),    # segments wider than the band
    (300, 1900, 1080)])
def test_mixed_walks(nverts, W, H, values, dtype):
    rng = np.random.default_rng(nverts + H)
    nlines = 1087
    xs = np.linspace(0.0, 1.0, nverts)
    ys = rng.normal(0, 1, (nlines, nverts))
    if values == "spikes":  # short segments, a long or clipped one now and then
        ys *= 0.01
        ys[rng.random(ys.shape) < 0.02] = 3.0
        ys[rng.random(ys.shape) < 0.02] = -1.99
    if values == "flat":    # one row, its ends on the view's bounds, or just off them
        ys = rng.choice([-2.0, 2.0, np.nextafter(2.0, 3), 0.0], ys.shape, p=[.1, .1, .1, .7])
    ys[rng.random(ys.shape) < 0.01] = np.nan
    ys = ys.astype(dtype)
    names = [f"y{j}" for j in range(nverts)]
    frame = dsa.DeviceFrame.from_block(names, torch.as_tensor(ys.T.copy(), device="cuda"))
    for xr in ((0.0, 1.0), (0.21, 0.64)):
        cvs = dsa.Canvas(W, H, x_range=xr, y_range=(-2.0, 2.0))
        got = cvs.line(frame, x=xs, y=names, agg=dsa.count(), axis=1).values
        view = G.view_for(W, H, xr, (-2.0, 2.0), yf32=dtype == np.float32)
        exp = oracle.lines_xconst(xs, ys.astype(np.float64), view, W, H)["count"]
        assert exp.sum() > 0
        np.testing.assert_array_equal(got, exp)
