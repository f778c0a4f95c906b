"""A pandas table of several pinned pieces on the device: every column kind, strided and
ragged-length columns, concurrent uploads; bytes equal to the host columns."""
from __future__ import annotations

from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pandas as pd
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import datashader_amd as dsa  # noqa: E402
from datashader_amd import _upload  # noqa: E402


def _frame(n, seed):
    rng = np.random.default_rng(seed)
    f32 = rng.normal(size=n).astype(np.float32)
    f32[::11] = np.nan
    wide = rng.integers(-9, 9, (n, 3))
    return pd.DataFrame({
        "x": rng.random(n), "y": f32, "i64": wide[:, 1], "i16": wide[:, 0].astype(np.int16),
        "u8": wide[:, 2].astype(np.uint8), "b": wide[:, 0] > 0, "z": rng.random((n, 2))[:, 1],
        "c": pd.Categorical.from_codes(rng.integers(-1, 5, n), list("abcde")),
        "s": pd.Series(["text"] * n)})


def _same(df, f):
    assert list(f.columns) == [c for c in df.columns if c != "s"]
    for c in f.columns:
        want = df[c].cat.codes.to_numpy() if c == "c" else df[c].to_numpy()
        got = f[c].cpu().numpy()
        assert got.dtype == want.dtype and got.tobytes() == np.ascontiguousarray(want).tobytes(), c


@pytest.mark.parametrize("n", [0, 1, 1000, 262_144, 524_288, 524_289, 1_700_003])
def test_columns(n):
    df = _frame(n, n)
    _same(df, dsa.DeviceFrame.from_pandas(df))


def test_threads():
    tables = [_frame(600_001 + 7 * i, i) for i in range(4)]

    def one(df):
        with torch.cuda.stream(torch.cuda.Stream()):
            return dsa.DeviceFrame.from_pandas(df)

    with ThreadPoolExecutor(4) as ex:
        for _ in range(2):
            for df, f in zip(tables, ex.map(one, tables)):
                _same(df, f)
    assert len(_upload._areas) <= _upload._KEPT
