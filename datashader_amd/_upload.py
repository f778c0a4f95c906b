"""Host columns to device memory through pinned pieces.

A copy from pageable memory runs at the rate of one host thread; here several threads copy
pieces of the columns into page-locked memory while the pieces before them go to the device
by DMA."""
from __future__ import annotations

import threading
from concurrent.futures import ThreadPoolExecutor

import numpy as np

# 8 pieces of 4 MiB: a call on 3M rows of three float64 columns 8.5 ms from pageable memory,
# 2.8 so
PIECE = 4 << 20
PIECES = 8
MIN_BYTES = 2 * PIECE
# Columns share a piece until it holds this much: a piece costs some 150 us of handing over
# between threads.  Larger columns keep pieces of their own, so that few columns still take
# several threads.
SHARED = 1 << 20
_KEPT = 2  # pinned areas (PIECES * PIECE bytes each) kept for later calls

_lock = threading.Lock()
_areas = []
_pool = None


def worth(nbytes, ncolumns):
    """Whether columns of ``nbytes`` in all are copied faster so than by the plain copy: from
    two pieces on if the columns hold 2 MiB each on average (four float64 columns of 250
    thousand rows, 8 MB: 534 us either way, eight of them 1121 -> 946).  Smaller columns cost
    more to hand over, so they need more of them: 1 MB columns 9 MB 0.58 -> 0.74 ms, 16 MB
    1.19 -> 1.40, 26 MB 1.89 -> 1.73; 0.3 MB columns 9 MB 0.93 -> 1.40 ms, 36 MB 5.6 either
    way; 0.08 MB columns 36 MB 11.6 -> 13.8.  So mean size squared times size of 32 MiB^3."""
    return nbytes >= MIN_BYTES and nbytes ** 3 >= ncolumns ** 2 * 32 * (1 << 20) ** 3


def _take():
    """A pinned area no other call uses, and the copying threads."""
    global _pool
    with _lock:
        if _pool is None:
            _pool = ThreadPoolExecutor(max_workers=PIECES, thread_name_prefix="dsa-upload")
        area = _areas.pop() if _areas else None
    if area is None:
        import torch
        area = torch.empty(PIECES * PIECE, dtype=torch.uint8, pin_memory=True)
    return area, _pool


def _give(area):
    with _lock:
        if len(_areas) < _KEPT:
            _areas.append(area)


def pieces(blocks):
    """How ``blocks`` (see ``upload``) go through the pinned area: per piece its copies into
    the area [(rows of an array, byte offset in the piece)] and its copies out of it
    [(block, first element, byte offset in the piece, elements)]."""
    out, ins, outs, used = [], [], [], 0
    for b, (arrays, _) in enumerate(blocks):
        size = arrays[0].dtype.itemsize
        used = -(-used // 16) * 16  # (every type's elements aligned)
        if used >= PIECE:
            out.append((ins, outs))
            ins, outs, used = [], [], 0
        for j, a in enumerate(arrays):
            at = 0
            while at < len(a):
                k = min(len(a) - at, (PIECE - used) // size)
                if k == 0:
                    out.append((ins, outs))
                    ins, outs, used = [], [], 0
                    continue
                ins.append((a[at:at + k], used))
                first = j * len(a) + at
                if outs and outs[-1][0] == b:  # (goes on where the last one ends)
                    outs[-1] = (b, outs[-1][1], outs[-1][2], outs[-1][3] + k)
                else:
                    outs.append((b, first, used, k))
                used += k * size
                at += k
            if used >= SHARED:
                out.append((ins, outs))
                ins, outs, used = [], [], 0
    if ins:
        out.append((ins, outs))
    return out


def _fill(host, ins):
    for src, at in ins:
        np.copyto(host[at:at + src.nbytes].view(src.dtype), src)


def upload(blocks):
    """Copy every (numpy arrays of one dtype and length, contiguous device tensor of that
    dtype with the arrays' elements one array after the other) of ``blocks``.  The tensors
    are complete when this returns, on every stream."""
    import torch
    area, pool = _take()
    host = area.numpy()
    work = pieces(blocks)
    flat = [t.view(-1) for _, t in blocks]
    stream = torch.cuda.current_stream(flat[0].device)
    jobs, done = [], []

    def stage(i):
        at = (i % PIECES) * PIECE
        jobs.append(pool.submit(_fill, host[at:at + PIECE], work[i][0]))

    try:
        for i in range(min(PIECES, len(work))):
            stage(i)
        for i, (_, outs) in enumerate(work):
            jobs[i].result()
            for b, first, at, k in outs:
                at += (i % PIECES) * PIECE
                dst = flat[b][first:first + k]
                dst.copy_(area[at:at + k * dst.element_size()].view(dst.dtype), non_blocking=True)
            ev = torch.cuda.Event()
            ev.record(stream)
            done.append(ev)
            # (two pieces' DMA stay queued while the one before them gives its memory back)
            if i >= 2 and i - 2 + PIECES < len(work):
                done[i - 2].synchronize()
                stage(i - 2 + PIECES)
    finally:  # no thread and no DMA uses the area when the next call takes it
        for f in jobs:
            f.cancel()
        for f in jobs:
            if not f.cancelled():
                f.exception()
        stream.synchronize()  # (not the last event: a piece that failed half-way has none)
        _give(area)
