"""The workspace of a statistics call (no GPU needed): the pass of squared deviations is
planned by itself, so one plane that fits tiles is tiled also where the planes of the first
pass together are beyond them."""
from __future__ import annotations

import pytest

from datashader_amd import _abi


def _size(W, H, planes, m2, val=_abi.F64):
    d = _abi.PointsDesc()
    d.n, d.x, d.y, d.val = 1_000_000, 256, 256, 256  # (addresses are not read)
    d.xy_dtype, d.val_dtype, d.strategy = _abi.F64, val, _abi.STRATEGY_AUTO
    v = _abi.View()
    v.sx = v.sy = v.xmax = v.ymax = 1.0
    v.width, v.height = W, H
    p = _abi.Planes()
    for k in planes:
        setattr(p, k, 256)
    lib = _abi.load()
    return int((lib.dsx_points_m2_workspace_size if m2 else lib.dsx_points_workspace_size)(d, v, p))


@pytest.mark.parametrize("W,H,first_tiled", [(700, 500, True), (4096, 4095, True),
                                             (4200, 4000, False), (8000, 8000, False)])
def test_m2_workspace_holds_a_tiled_pass(W, H, first_tiled):
    stats = ("countv", "sum", "min", "max", "mean")
    one, first = _size(W, H, ("sum",), False), _size(W, H, stats, False)
    assert (first > 1 << 20) == first_tiled and one > 1 << 20
    assert _size(W, H, stats, True) >= max(one if not first_tiled else 0, first)
