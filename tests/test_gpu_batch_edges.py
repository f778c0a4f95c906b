"""The batched aggregation kernel where it can go wrong: sets shorter than a step of its
threads, steps that end inside a lattice row, rows that all meet in one pixel or one lattice
cell, tiles of one pixel, tiles over many lattice rows, split tiles, every workgroup size.
Counts exact; the values are small whole numbers, so their float64 sums are exact in any order,
and a mean is one division of exact numbers."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from oracle import closed_forms as cf

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import datashader_amd as dsa  # noqa: E402
from datashader_amd import batching, serving  # noqa: E402


def _check(x, y, v, grid, views, threads, knobs, count_only=False):
    tx, ty, tv = (torch.as_tensor(a, device="cuda") for a in (x, y, v))
    index = serving.PointIndex(tx, ty, None if count_only else tv, grid=grid,
                               extent=((0.0, 1.0), (0.0, 1.0)))
    agg = dsa.count() if count_only else dsa.summary(c=dsa.count(), cv=dsa.count("v"),
                                                     s=dsa.sum("v"), m=dsa.mean("v"))
    tuning = batching.Tuning(threads=threads)
    if knobs is not None:
        tuning.DEFAULT = knobs
    server = batching.BatchServer(index, agg=agg, engines=1, max_batch=8, tuning=tuning)
    reqs = [serving.Request(xr, yr, W, H, agg) for W, H, xr, yr in views]
    got = server.serve(reqs, realtime=False, keep_results=True)["results"]
    for (W, H, xr, yr), res in zip(views, got):
        sx, sy = W / (xr[1] - xr[0]), H / (yr[1] - yr[0])
        view = oracle.View(sx, -xr[0] * sx, sy, -yr[0] * sy, xr[0], xr[1], yr[0], yr[1])
        bins = cf.point_bins(x.astype(np.float64), y.astype(np.float64), view, W, H)
        if count_only:
            np.testing.assert_array_equal(res.values, cf.count(bins, W, H))
            continue
        np.testing.assert_array_equal(res["c"].values, cf.count(bins, W, H))
        np.testing.assert_array_equal(res["cv"].values, cf.count(bins, W, H, v))
        np.testing.assert_array_equal(res["s"].values, cf.sum_nan(bins, v, W, H))
        np.testing.assert_array_equal(res["m"].values, cf.mean(bins, v, W, H))
    server.close()


VIEWS = [(64, 48, (0.0, 1.0), (0.0, 1.0)), (1, 1, (0.0, 1.0), (0.0, 1.0)),
         (300, 200, (0.4, 0.6), (0.1, 0.9)), (33, 777, (-0.5, 1.5), (0.25, 0.5))]


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 255, 256, 257, 1025, 70_001])
@pytest.mark.parametrize("threads", [256, 512, 1024])
def test_row_counts(n, threads):
    rng = np.random.default_rng(n)
    x, y = rng.uniform(0, 1, (2, n)).astype(np.float32)
    v = rng.integers(-50, 50, n).astype(np.float32)
    v[::7] = np.nan
    _check(x, y, v, 64, VIEWS, threads, None)
    _check(x, y, v, 64, VIEWS[:2], threads, None, count_only=True)


@pytest.mark.parametrize("spread", ["one", "two", "cell"])
@pytest.mark.parametrize("cells,tile_h,part", [(1, 1, 1 << 18), (300, 8, 1000), (1260, 32, 300),
                                               (2520, 64, 1 << 18), (0, 64, 5000)])
def test_rows_that_meet(spread, cells, tile_h, part):
    """Whole steps in one pixel, steps over two pixels, steps over one lattice cell."""
    rng = np.random.default_rng(cells)
    n = 20_011
    x = np.full(n, 0.501, np.float32)
    y = np.full(n, 0.25, np.float32)
    if spread == "two":
        x[n // 3:] = 0.517
    if spread == "cell":
        x = (0.5 + rng.uniform(0, 1 / 16, n)).astype(np.float32)
        y = (0.25 + rng.uniform(0, 1 / 16, n)).astype(np.float32)
    v = rng.integers(-50, 50, n).astype(np.float32)
    v[rng.random(n) < 0.01] = np.nan
    views = VIEWS[1:] if cells == 1 else VIEWS
    if cells == 1:  # (a tile a pixel: small canvases)
        views = [(9, 7, (0.0, 1.0), (0.0, 1.0)), (1, 1, (0.0, 1.0), (0.0, 1.0))]
    _check(x, y, v, 16, views, 1024, {"tile_h": tile_h, "tile_cells": cells, "part_rows": part})


@pytest.mark.parametrize("grid", [255, 256, 257, 2048])
def test_tiles_over_many_lattice_rows(grid):
    rng = np.random.default_rng(grid)
    n = 50_000
    x, y = rng.uniform(0, 1, (2, n)).astype(np.float32)
    v = rng.integers(-50, 50, n).astype(np.float32)
    _check(x, y, v, grid, VIEWS, 512, {"tile_h": 1000, "tile_cells": 0, "part_rows": 777})
