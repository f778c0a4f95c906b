"""The fixed-point walk of short line segments (dsx_lines.hip box_walk) against the
reference's error term (line.py:986-1031), over every segment shape it is used for."""
import numpy as np
import pytest


@pytest.mark.parametrize("ulp", [-1, 0, 1])  # the hardware reciprocal is within one ulp
def test_fixed_point_minor_axis_equals_bresenham(ulp):
    f32 = np.float32
    for n in range(1, 256):
        m = np.arange(n + 1, dtype=np.int64)
        i = np.arange(1, n + 1, dtype=np.int64)[:, None]
        rn = f32(1.0) / f32(n)
        if ulp:
            rn = np.nextafter(rn, f32(2.0 if ulp > 0 else 0.0), dtype=f32)
        slope = (m.astype(f32) * rn * f32(1048576.0)).astype(np.int64)
        quarter = int(rn * f32(262144.0))
        for b in (0, 1):  # 1: the major axis runs backwards
            moved = (524288 + (quarter if b == 0 else -quarter) + i * slope) >> 20
            # err >= 0 && (err || i > 0), err halved: 2m - n, then + 2m - 2n per minor move
            err = 2 * m - n - b
            want = np.zeros((n, n + 1), np.int64)
            at = np.zeros(n + 1, np.int64)
            for k in range(n):
                both = err >= 0
                at = at + both
                err = err + np.where(both, 2 * (m - n), 2 * m)
                want[k] = at
            np.testing.assert_array_equal(moved, want)
            assert moved.max() < 4096 and (slope <= 1 << 20).all()
