"""How columns are cut into pinned pieces (datashader_amd/_upload.py): every element once, in
bounds, and few pieces for many small columns."""
from __future__ import annotations

import numpy as np
import pytest

from datashader_amd import _upload


def _blocks(shapes, rng):
    out = []
    for dt, ncols, n in shapes:
        a = rng.integers(0, 100, (ncols, n)).astype(dt)
        if ncols > 1:
            a = np.asfortranarray(a)  # (columns of a row-major table: strided)
        out.append((list(a), np.full(ncols * n, 101).astype(dt)))
    return out


@pytest.mark.parametrize("shapes", [
    [("f8", 1, 1_100_003)], [("f8", 3, 350_000)], [("f4", 256, 10_001)], [("f8", 300, 333)],
    [("i1", 1, 5), ("i8", 1, 524_287), ("b1", 1, 7), ("f4", 2, 1_048_577), ("f8", 2, 3)],
    [("i1", 1, (4 << 20) - 3), ("f8", 1, 9)], [("i1", 1, 4 << 20), ("i2", 1, 9)],
    [("u1", 1, 12 << 20), ("f8", 1, 0), ("f4", 3, 1)]])
def test_pieces_cover_every_element_once(shapes):
    blocks = _blocks(shapes, np.random.default_rng(1))
    work = _upload.pieces(blocks)
    area = np.empty(_upload.PIECE, np.uint8)
    for ins, outs in work:
        area[:] = 0xEE
        _upload._fill(area, ins)
        for b, first, at, k in outs:
            flat = blocks[b][1]
            assert at % flat.itemsize == 0 and at + k * flat.itemsize <= _upload.PIECE
            flat[first:first + k] = area[at:at + k * flat.itemsize].view(flat.dtype)
    for arrays, flat in blocks:
        np.testing.assert_array_equal(flat, np.concatenate(arrays))
    assert sum(k for _, outs in work for *_, k in outs) == sum(c * n for _, c, n in shapes)


@pytest.mark.parametrize("ncols,n", [(256, 10_000), (5000, 300), (60, 20_000), (3, 1_000_000)])
def test_small_columns_share_pieces(ncols, n):
    work = _upload.pieces(_blocks([("f8", ncols, n)], np.random.default_rng(0)))
    assert len(work) <= ncols * n * 8 // _upload.SHARED + 1


def test_many_small_columns_keep_the_plain_copy():
    assert _upload.worth(3 * 8 * 350_000, 3) and _upload.worth(8 << 20, 1)
    assert not _upload.worth((8 << 20) - 1, 1)
    for ncols, n in ((256, 10_000), (500, 3000), (5000, 300), (60, 20_000), (9, 125_000), (15, 137_500)):
        assert not _upload.worth(8 * ncols * n, ncols)
