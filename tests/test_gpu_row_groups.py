"""The scans' grouped row loads at the ends of a table and of a chunk and at unaligned
columns: every row counted once, none from beyond the table.  Against the oracle's closed
forms; counts and selected rows exact, and the values small whole numbers, so that their
float64 sums are exact in any order."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import closed_forms as cf

import golden_utils as G

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import datashader_amd as dsa  # noqa: E402
from datashader_amd import _abi, backend  # noqa: E402

W, H = 512, 300


@pytest.fixture(params=[_abi.STRATEGY_WINDOW, _abi.STRATEGY_TILES], ids=["window", "tiles"])
def strategy(request):
    backend.FORCE_STRATEGY = request.param
    yield
    backend.FORCE_STRATEGY = None


def _column(a, off):
    """The array on the device, its first element `off` elements past an allocation's start."""
    t = torch.empty(len(a) + off + 1, dtype=getattr(torch, str(a.dtype)), device="cuda")
    t[off:off + len(a)] = torch.from_numpy(a).cuda()
    return t[off:off + len(a)]


def _frame(n, off, ct, vt, rng):
    x, y = rng.random((2, n)).astype(ct)
    v = rng.integers(-9, 10, n).astype(vt)
    v[::11] = np.nan
    cat = rng.integers(-1, 5, n).astype(np.int8)  # (-1 wraps to the last, 4 is dropped)
    f = dsa.DeviceFrame({"x": _column(x, off), "y": _column(y, off), "v": _column(v, off),
                         "cat": _column(cat, off)}, categories={"cat": list("abcd")})
    return x, y, v, cat, f


SIZES = [1, 2, 3, 4, 5, 6, 7, 4095, 4096, 4097, 4098, 6143, 6145, 8193, 70_002, 70_003]


@pytest.mark.parametrize("off", [0, 1, 3])
@pytest.mark.parametrize("ct,vt", [(np.float32, np.float32), (np.float64, np.float64),
                                   (np.float32, np.float64), (np.float64, np.float32)])
def test_points(strategy, ct, vt, off):
    rng = np.random.default_rng(off)
    view = G.view_for(W, H, (0.1, 0.9), (0.0, 1.0))
    cvs = dsa.Canvas(W, H, x_range=(0.1, 0.9), y_range=(0.0, 1.0))
    for n in SIZES:
        x, y, v, cat, f = _frame(n, off, ct, vt, rng)
        b = cf.point_bins(x, y, view, W, H)
        got = cvs.points(f, "x", "y", dsa.summary(c=dsa.count(), s=dsa.sum("v"), m=dsa.mean("v")))
        np.testing.assert_array_equal(got["c"].values, cf.count(b, W, H), err_msg=str(n))
        np.testing.assert_array_equal(got["s"].values, cf.sum_nan(b, v, W, H), err_msg=str(n))
        np.testing.assert_array_equal(got["m"].values, cf.mean(b, v, W, H), err_msg=str(n))
        np.testing.assert_array_equal(cvs.points(f, "x", "y").values, cf.count(b, W, H))
        k = np.where(cat < 0, cat + 4, cat).astype(np.int64)
        kb = np.where((b >= 0) & (k < 4), b * 4 + k, -1)
        got = cvs.points(f, "x", "y", dsa.by("cat", dsa.count())).values
        np.testing.assert_array_equal(got.reshape(-1), cf.count(kb, 4 * W, H).reshape(-1))
        got = cvs.points(f, "x", "y", dsa.by("cat", dsa.mean("v"))).values
        np.testing.assert_array_equal(got.reshape(-1), cf.mean(kb, v, 4 * W, H).reshape(-1))


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("ct,vt", [(np.float32, np.float32), (np.float64, np.float64)])
def test_selected_rows(ct, vt, off):
    rng = np.random.default_rng(off + 7)
    view = G.view_for(W, H, (0.1, 0.9), (0.0, 1.0))
    cvs = dsa.Canvas(W, H, x_range=(0.1, 0.9), y_range=(0.0, 1.0))
    for n in SIZES:
        x, y, v, _, f = _frame(n, off, ct, vt, rng)
        b = cf.point_bins(x, y, view, W, H)
        ok = np.flatnonzero((b >= 0) & ~np.isnan(v))
        first = np.full(W * H, -1, np.int64)
        last = first.copy()
        first[b[ok[::-1]]] = ok[::-1]
        last[b[ok]] = ok
        order = ok[np.lexsort((ok, -v[ok]))]
        top = np.full(W * H, -1, np.int64)
        top[b[order[::-1]]] = order[::-1]
        for red, want in ((dsa.first("v"), first), (dsa.last("v"), last)):
            exp = np.where(want < 0, np.nan, v[want].astype(np.float64)).reshape(H, W)
            np.testing.assert_array_equal(cvs.points(f, "x", "y", red).values, exp, err_msg=str(n))
        got = cvs.points(f, "x", "y", dsa.where(dsa.max("v"))).values
        np.testing.assert_array_equal(got, top.reshape(H, W), err_msg=str(n))
        got = cvs.points(f, "x", "y", dsa.max_n("v", n=2)).values[:, :, 0]
        exp = np.where(top < 0, np.nan, v[top].astype(np.float64)).reshape(H, W)
        np.testing.assert_array_equal(got, exp, err_msg=str(n))
