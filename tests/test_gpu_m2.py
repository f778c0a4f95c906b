"""var / std with their planes in one call: under each strategy and AUTO, split tiles, a
canvas that fits a window, canvases beyond the tiles, categories and NaN values.  The
squared deviations are taken from the same finished means as the two-call form's, so only
the order of the float64 additions differs: 1e-9 relative, the tolerance var / std have
here for float64 values (1e-5 for float32)."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import closed_forms as cf

import golden_utils as G

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import datashader_amd as dsa  # noqa: E402
from datashader_amd import _abi, backend  # noqa: E402


@pytest.mark.parametrize("strategy", [None, _abi.STRATEGY_WINDOW, _abi.STRATEGY_TILES],
                         ids=["auto", "window", "tiles"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("spread,W,H,n", [("uniform", 700, 500, 300_001), ("hot", 700, 500, 300_001),
                                          ("one", 400, 300, 50_000), ("uniform", 30, 20, 5_000),
                                          ("uniform", 600, 400, 3), ("uniform", 600, 400, 0),
                                          ("uniform", 8200, 8200, 20_000)])
def test_std_and_planes(strategy, dt, spread, W, H, n):
    if n == 20_000 and strategy is not None:
        pytest.skip("a canvas beyond the tiles has one way")
    rng = np.random.default_rng(n)
    x, y = rng.random((2, n))
    if spread == "hot":
        hot = rng.random(n) < 0.9
        x[hot], y[hot] = 0.5 + 0.01 * rng.standard_normal((2, int(hot.sum())))
    if spread == "one":  # one tile holds nearly all rows: it is split
        x, y = 0.5 + x / 50, np.full(n, 0.5)
    x, y = x.astype(dt), y.astype(dt)
    v = rng.normal(100, 3, n).astype(dt)
    v[::13] = np.nan
    f = dsa.DeviceFrame({k: torch.from_numpy(a).cuda() for k, a in (("x", x), ("y", y), ("v", v))})
    cvs = dsa.Canvas(W, H, x_range=(0.0, 1.0), y_range=(0.0, 1.0))
    b = cf.point_bins(x, y, G.view_for(W, H, (0.0, 1.0), (0.0, 1.0)), W, H)
    var = cf.var2pass(b, v, W, H)
    backend.FORCE_STRATEGY = strategy
    try:
        for _ in range(2):  # (AUTO: the second call passes the strategy the first picked)
            got = cvs.points(f, "x", "y", dsa.summary(n=dsa.count("v"), lo=dsa.min("v"),
                                                      m=dsa.mean("v"), s=dsa.std("v"), q=dsa.var("v")))
            torch.cuda.synchronize()
            np.testing.assert_array_equal(got["n"].values, cf.count(b, W, H, v))
            tol = 1e-5 if dt is np.float32 else 1e-9
            for k, want in (("s", np.sqrt(var)), ("q", var)):
                a = got[k].values
                np.testing.assert_array_equal(np.isnan(a), np.isnan(want))
                ok = ~np.isnan(want)
                np.testing.assert_allclose(a[ok], want[ok], rtol=tol, atol=1e-18)
            np.testing.assert_allclose(got["m"].values, cf.mean(b, v, W, H), rtol=1e-12)
    finally:
        backend.FORCE_STRATEGY = None
