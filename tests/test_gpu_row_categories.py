"""The scans' grouped row loads with categorizer columns of every width: at the ends of a table
and of a chunk, at unaligned columns, and over several chunks a workgroup (the loaders' register
sets change roles).  Against closed forms; counts exact, and the values small whole numbers, so
that their float64 sums are exact in any order and a mean is one division of exact numbers."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import closed_forms as cf

import golden_utils as G

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import datashader_amd as dsa  # noqa: E402
from datashader_amd import _abi, backend  # noqa: E402

W, H = 211, 130
XR, YR = (0.1, 0.9), (0.0, 1.0)


@pytest.fixture(params=[_abi.STRATEGY_WINDOW, _abi.STRATEGY_TILES], ids=["window", "tiles"])
def strategy(request):
    backend.FORCE_STRATEGY = request.param
    yield
    backend.FORCE_STRATEGY = None


def _column(a, off):
    t = torch.empty(len(a) + off + 1, dtype=getattr(torch, str(a.dtype)), device="cuda")
    t[off:off + len(a)] = torch.from_numpy(a).cuda()
    return t[off:off + len(a)]


def _keys(kind, n, rng):
    """(column, categorizer, category of every row or -1, categories)"""
    how, dt = kind.split("-")
    dt = np.dtype(dt)
    if how == "codes":
        k = rng.integers(-1, 5, n).astype(dt)  # (-1 wraps to the last, 4 is dropped)
        w = k.astype(np.int64)
        return k, "k", np.where(w < 0, w + 4, np.where(w < 4, w, -1)), 4
    k = rng.integers(0 if dt.kind == "u" else -100, 100, n)
    if how == "mod":
        return k.astype(dt), dsa.category_modulo("k", 5, 3), (k - 3) % 5, 5
    if dt.kind == "f":
        k = k + 0.25
        k[::7] = np.nan
    k = k.astype(dt)
    b = np.floor((np.nan_to_num(k.astype(np.float64)) + 40.0) / 16.0).astype(np.int64)
    cat = np.where(b < 0, 0, np.where(b >= 5, 5, b))  # (values above are not included: bin 5)
    cat = np.where(np.isnan(k.astype(np.float64)), 5, cat)
    return k, dsa.category_binning("k", -40, 40, 5, include_over=False), cat, 6


def _check(kind, n, ct, off, rng):
    x, y = rng.random((2, n)).astype(ct)
    v = rng.integers(-9, 10, n).astype(ct)
    v[::11] = np.nan
    k, by, cat, ncat = _keys(kind, n, rng)
    f = dsa.DeviceFrame({c: _column(a, off) for c, a in (("x", x), ("y", y), ("v", v), ("k", k))},
                        categories={"k": list("abcd")} if by == "k" else None)
    cvs = dsa.Canvas(W, H, x_range=XR, y_range=YR)
    b = cf.point_bins(x, y, G.view_for(W, H, XR, YR), W, H)
    kb = np.where((b >= 0) & (cat >= 0), b * ncat + cat, -1)
    got = cvs.points(f, "x", "y", dsa.by(by, dsa.count())).values
    np.testing.assert_array_equal(got.reshape(-1), cf.count(kb, ncat * W, H).reshape(-1))
    got = cvs.points(f, "x", "y", dsa.by(by, dsa.mean("v"))).values
    np.testing.assert_array_equal(got.reshape(-1), cf.mean(kb, v, ncat * W, H).reshape(-1))


KINDS = ["codes-uint8", "codes-int16", "codes-int32", "codes-int64", "mod-int8", "mod-uint8",
         "mod-int16", "mod-int32", "mod-int64", "bin-int8", "bin-uint8", "bin-int32", "bin-float32",
         "bin-float64"]


@pytest.mark.parametrize("ct", [np.float32, np.float64])
@pytest.mark.parametrize("kind", KINDS)
def test_ends(strategy, kind, ct):
    rng = np.random.default_rng(len(kind))
    for n in (1, 2, 3, 4, 5, 7, 4095, 4097, 4098, 8193, 70_003):
        for off in (0, 1, 3):
            _check(kind, n, ct, off, rng)


@pytest.mark.parametrize("n", [2_100_003, 3_200_001])
@pytest.mark.parametrize("kind", ["codes-int32", "codes-int64", "mod-int8", "bin-float64"])
@pytest.mark.parametrize("ct", [np.float32, np.float64])
def test_several_chunks_a_workgroup(strategy, kind, n, ct):
    _check(kind, n, ct, 1, np.random.default_rng(n))


@pytest.mark.parametrize("n", [5, 8193, 3_200_001])
@pytest.mark.parametrize("kind", ["codes-int16", "codes-int64", "bin-float64"])
@pytest.mark.parametrize("ct,vt", [(np.float64, np.float64), (np.float32, np.float64),
                                   (np.float64, np.float32)])
def test_selected_rows(kind, n, ct, vt):
    """The first, the last and the largest value's row of each category (the row-index scans)."""
    rng = np.random.default_rng(n + 1)
    x, y = rng.random((2, n)).astype(ct)
    v = rng.integers(-99, 100, n).astype(vt)  # (ties: the first row is taken)
    v[::11] = np.nan
    k, by, cat, ncat = _keys(kind, n, rng)
    f = dsa.DeviceFrame({c: _column(a, 1) for c, a in (("x", x), ("y", y), ("v", v), ("k", k))},
                        categories={"k": list("abcd")} if by == "k" else None)
    cvs = dsa.Canvas(W, H, x_range=XR, y_range=YR)
    b = cf.point_bins(x, y, G.view_for(W, H, XR, YR), W, H)
    ok = np.flatnonzero((b >= 0) & (cat >= 0) & ~np.isnan(v))
    cell = b[ok] * ncat + cat[ok]
    first, last, top = (np.full(W * H * ncat, -1, np.int64) for _ in range(3))
    first[cell[::-1]] = ok[::-1]
    last[cell] = ok
    order = np.lexsort((ok, -v[ok]))[::-1]
    top[cell[order]] = ok[order]
    for red, want in ((dsa.first("v"), first), (dsa.last("v"), last)):
        exp = np.where(want < 0, np.nan, v[want].astype(np.float64)).reshape(H, W, ncat)
        np.testing.assert_array_equal(cvs.points(f, "x", "y", dsa.by(by, red)).values, exp)
    got = cvs.points(f, "x", "y", dsa.by(by, dsa.where(dsa.max("v")))).values
    np.testing.assert_array_equal(got, top.reshape(H, W, ncat))
