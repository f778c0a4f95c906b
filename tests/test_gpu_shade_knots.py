"""The colour pass around the number of knots that LDS holds (512), with one colour and
with value ranges whose knots are not evenly representable: linear and eq_hist equal to
the oracle (pure IEEE arithmetic in both)."""
from __future__ import annotations

import numpy as np
import pytest

import datashader_amd as dsa
import datashader_amd.transfer_functions as tf
from golden_utils import shade_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("how", ["linear", "eq_hist"])
@pytest.mark.parametrize("dtype", ["u4", "i8", "f4", "f8"])
@pytest.mark.parametrize("nk", [1, 2, 255, 511, 512, 513, 1500])
def test_knots(nk, dtype, how):
    import torch
    rng = np.random.default_rng(nk)
    if dtype in ("u4", "i8"):
        data = rng.integers(0, 70_000 if nk % 2 else 900, (93, 211)).astype(dtype)
    else:
        data = (1e-3 * rng.normal(size=(93, 211)) + 7).astype(dtype)
        data[rng.random(data.shape) < 0.2] = np.nan
    t = torch.from_numpy(data.view(np.int32) if dtype == "u4" else data).cuda()
    plane = dsa.DataArray(t.view(torch.uint32) if dtype == "u4" else t, dims=["y", "x"],
                          coords={"x": np.arange(211), "y": np.arange(93)})
    cmap = [tuple(int(v) for v in c) for c in rng.integers(0, 256, (nk, 3))]
    for kw in ({"cmap": cmap, "how": how}, {"cmap": "red", "how": how, "min_alpha": nk % 200}):
        np.testing.assert_array_equal(np.asarray(tf.shade(plane, **kw).values, np.uint32),
                                      shade_oracle(data, kw))
