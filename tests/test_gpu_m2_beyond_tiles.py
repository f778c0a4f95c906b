"""var / std where the first pass's planes are beyond the tiles (global atomics) and the plane of
squared deviations is not (a tiled pass): every strategy that pass can take, rows spread out and
in one place.  The tolerance of var / std for float64 values (1e-9 relative: the order of the
float64 additions differs)."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import closed_forms as cf

import golden_utils as G

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import datashader_amd as dsa  # noqa: E402
from datashader_amd import _abi, backend  # noqa: E402

W, H = 4200, 4000


@pytest.mark.parametrize("strategy", [None, _abi.STRATEGY_WINDOW, _abi.STRATEGY_TILES],
                         ids=["auto", "window", "tiles"])
@pytest.mark.parametrize("spread", ["uniform", "hot"])
def test_std(spread, strategy):
    n = 300_001
    rng = np.random.default_rng(n)
    x, y = rng.random((2, n))
    if spread == "hot":
        x, y = 0.5 + x / 100, 0.5 + y / 100
    v = rng.normal(100, 3, n)
    v[::13] = np.nan
    f = dsa.DeviceFrame({k: torch.from_numpy(a).cuda() for k, a in (("x", x), ("y", y), ("v", v))})
    cvs = dsa.Canvas(W, H, x_range=(0.0, 1.0), y_range=(0.0, 1.0))
    b = cf.point_bins(x, y, G.view_for(W, H, (0.0, 1.0), (0.0, 1.0)), W, H)
    want = np.sqrt(cf.var2pass(b, v, W, H))
    agg = dsa.summary(n=dsa.count("v"), lo=dsa.min("v"), hi=dsa.max("v"), t=dsa.sum("v"),
                      s=dsa.std("v"))
    backend.FORCE_STRATEGY = strategy
    try:
        for _ in range(2):
            got = cvs.points(f, "x", "y", agg)
            np.testing.assert_array_equal(got["n"].values, cf.count(b, W, H, v))
            a = got["s"].values
            np.testing.assert_array_equal(np.isnan(a), np.isnan(want))
            ok = ~np.isnan(want)
            np.testing.assert_allclose(a[ok], want[ok], rtol=1e-9, atol=1e-18)
    finally:
        backend.FORCE_STRATEGY = None
