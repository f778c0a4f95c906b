"""Canvases whose buckets fit the tile strategy's scan only with tiles of twice the usual
size, and their neighbours below and above: mean and extremes under each strategy, the
second call with the first one's stored window.  Counts and extremes are equal, means to
1e-12 (the order of float64 additions)."""
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
@pytest.mark.parametrize("spread", ["uniform", "hot"])
@pytest.mark.parametrize("dt,W,H", [(np.float64, 1600, 900), (np.float64, 1800, 1000),
                                    (np.float64, 2600, 1500), (np.float32, 1920, 1080),
                                    (np.float32, 3001, 1799)])
def test_planes(strategy, spread, dt, W, H):
    n = 400_003
    rng = np.random.default_rng(W)
    x, y = rng.random((2, n))
    if spread == "hot":
        hot = rng.random(n) < 0.9
        x[hot], y[hot] = 0.5 + 0.005 * rng.standard_normal((2, int(hot.sum())))
    x, y = x.astype(dt), y.astype(dt)
    v = rng.normal(100, 3, n).astype(dt)
    v[::17] = np.nan
    f = dsa.DeviceFrame({k: torch.from_numpy(a).cuda() for k, a in (("x", x), ("y", y), ("v", v))})
    cvs = dsa.Canvas(W, H, x_range=(0.0, 1.0), y_range=(0.0, 1.0))
    b = cf.point_bins(x, y, G.view_for(W, H, (0.0, 1.0), (0.0, 1.0)), W, H)
    backend.FORCE_STRATEGY = strategy
    try:
        for agg in (dsa.summary(n=dsa.count("v"), lo=dsa.min("v"), hi=dsa.max("v"), m=dsa.mean("v")),
                    dsa.summary(c=dsa.count(), n=dsa.count("v"), m=dsa.mean("v"))):
            for _ in range(2):
                got = cvs.points(f, "x", "y", agg)
                torch.cuda.synchronize()
                np.testing.assert_array_equal(got["n"].values, cf.count(b, W, H, v))
                np.testing.assert_allclose(got["m"].values, cf.mean(b, v, W, H), rtol=1e-12)
                if "lo" in got:
                    lo, hi = cf.minmax(b, v, W, H)
                    np.testing.assert_array_equal(got["lo"].values, lo)
                    np.testing.assert_array_equal(got["hi"].values, hi)
                else:
                    np.testing.assert_array_equal(got["c"].values, cf.count(b, W, H))
    finally:
        backend.FORCE_STRATEGY = None


@pytest.mark.parametrize("W,H", [(1000, 700), (2600, 1500)], ids=["means-in-lds", "means-gathered"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_std_over_tiles(dt, W, H):
    """The second tile pass with its tile's means in LDS, and where they do not fit there."""
    n = 300_001
    rng = np.random.default_rng(H)
    x, y = rng.random((2, n)).astype(dt)
    v = rng.normal(100, 3, n).astype(dt)
    v[::17] = np.nan
    f = dsa.DeviceFrame({k: torch.from_numpy(a).cuda() for k, a in (("x", x), ("y", y), ("v", v))})
    cvs = dsa.Canvas(W, H, x_range=(0.0, 1.0), y_range=(0.0, 1.0))
    b = cf.point_bins(x, y, G.view_for(W, H, (0.0, 1.0), (0.0, 1.0)), W, H)
    backend.FORCE_STRATEGY = _abi.STRATEGY_TILES
    try:
        got = cvs.points(f, "x", "y", dsa.summary(m=dsa.mean("v"), s=dsa.std("v")))
        torch.cuda.synchronize()
    finally:
        backend.FORCE_STRATEGY = None
    want = np.sqrt(cf.var2pass(b, v, W, H))
    ok = ~np.isnan(want)
    np.testing.assert_array_equal(np.isnan(got["s"].values), ~ok)
    # (as for std elsewhere: 1e-9 for float64 values, 1e-5 for float32)
    np.testing.assert_allclose(got["s"].values[ok], want[ok], rtol=1e-5 if dt is np.float32 else 1e-9, atol=1e-9)
    np.testing.assert_allclose(got["m"].values, cf.mean(b, v, W, H), rtol=1e-12)
