"""Host set-up of the coarse correction on row patterns that do not come from
a box: a block's rows may reach at most as many neighbour blocks as the sweep
kernels' LDS teams of eight list entries hold; beyond, the correction is
refused at set-up."""
import ctypes as C

import numpy as np
import pytest

KCQ = 32


def layout(rp, cols, pc_block, part=None):
    """(rc, message, sizes, block of each row, group of each block, overlaps)."""
    from tdycore_amd import _lib
    L = _lib.load()
    rp, cols = (np.ascontiguousarray(a, dtype=np.int32) for a in (rp, cols))
    nc = len(rp) - 1
    sizes, blk, grp = np.zeros(5, np.int32), np.full(nc, -1, np.int32), np.full(nc, -1, np.int32)
    gov = np.full(nc * 128, -1, np.int32)
    p = None if part is None else np.ascontiguousarray(part, dtype=np.int32)
    ptr = lambda a: None if a is None else a.ctypes.data_as(C.c_void_p)  # noqa: E731
    rc = L.tdyhip_test_coarse_layout(ptr(rp), ptr(cols), nc, pc_block, ptr(p), ptr(sizes), ptr(blk), ptr(grp), ptr(gov))
    return rc, L.tdyhip_last_error().decode(), sizes, blk, grp, gov


def _scattered(block, reach, rows=None):
    """32 blocks of `block` rows; of each block the first `rows` rows couple
    to the same row of `reach` other blocks (and to themselves)."""
    nb = 32
    i = np.arange(block * nb)
    b, r = i // block, i % block
    near = [np.where((r < (block if rows is None else rows)), (((b + d) % nb) * block + r), i)
            for d in list(range(0, reach // 2 + 1)) + list(range(-((reach + 1) // 2), 0))]
    cols = [np.unique(c) for c in np.stack(near, axis=1)]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])])
    return rp, np.concatenate(cols), b


@pytest.mark.parametrize("block", [64, 256, 512])
def test_rows_scattered_over_every_neighbour_are_refused(block):
    rp, cols, part = _scattered(block, 31)
    assert np.diff(rp).max() == 32
    teams = 31 * block // 8
    assert teams > block * 27 // 8 + KCQ or block == 64
    rc, msg, sizes, *_ = layout(rp, cols, block, part)
    if teams <= block * 27 // 8 + KCQ:
        assert rc == 0 and sizes[4] == teams
    else:
        assert rc == 1 and "neighbour blocks" in msg


@pytest.mark.parametrize("block", [64, 256, 512])
def test_the_most_teams_that_fit(block):
    """27 entries in 27 blocks, and the last row count of 32 entries that fits."""
    rp, cols, part = _scattered(block, 26)
    rc, _, sizes, *_ = layout(rp, cols, block, part)
    assert rc == 0 and sizes[4] == 26 * block // 8
    rows = min(block, 8 * ((block * 27 // 8 + KCQ) // 31))
    rp, cols, part = _scattered(block, 31, rows)
    rc, _, sizes, *_ = layout(rp, cols, block, part)
    assert rc == 0 and sizes[4] == 31 * rows // 8 <= block * 27 // 8 + KCQ
    if rows < block:
        rp, cols, part = _scattered(block, 31, rows + 1)
        assert layout(rp, cols, block, part)[0] == 1


def test_rows_of_more_than_32_entries_are_refused():
    n = 33
    rp, cols = np.arange(n + 1) * n, np.tile(np.arange(n), n)
    rc, msg, *_ = layout(rp, cols, 64, np.arange(n) // 2)
    assert rc == 1 and "32 entries" in msg
