"""Column bounds at every alignment of the first row and around whole pieces and steps of
the 16-byte loads, with missing values: equal to numpy's nanmin / nanmax."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from datashader_amd import _device as dev  # noqa: E402


@pytest.mark.parametrize("off", [0, 1, 2, 3])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("n", [0, 1, 2, 3, 4, 5, 255, 256, 257, 4099, 524_288 * 4 + 5, 4_200_001, 9_000_003])
def test_bounds(n, dt, off):
    rng = np.random.default_rng(n + off)
    a = rng.normal(0, 100, n + off).astype(dt)
    a[::7] = np.nan
    if n > 3:  # the extremes in the first, last and middle rows in turn
        a[off], a[-1], a[off + n // 2] = -1e6 + off, 1e6, np.nan
    col = torch.from_numpy(a).cuda()[off:]
    lo, hi = dev.bounds(col)
    b = a[off:]
    b = b[~np.isnan(b)]
    if len(b):
        assert (lo, hi) == (float(b.min()), float(b.max()))
    else:
        assert not (np.isfinite(lo) and np.isfinite(hi))
