"""The hub block's selections on the device against numpy: level counts, the
rows and columns in a range, and the list of 64-nonzero tiles in the block."""
import ctypes

import numpy as np
import pytest

import powersparse_amd as ps
from powersparse_amd import _native
from gpu_util import say, setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 256, 257, 4097, 300000])
def test_levels_and_select(n):
    setup()
    say(f"hub select n={n}")
    rng = np.random.default_rng(n)
    deg = (2.0 ** rng.uniform(0, 14, n)).astype(np.int64) * (rng.random(n) < 0.7)
    deg = np.minimum(deg, ((1 << 31) - 1) // n)
    if n == 1:
        deg[:] = (1 << 31) - 1  # the top level
    row_ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    cnt = rng.permutation(deg).astype(np.int32)
    d_ptr, d_cnt = ps.DeviceBuffer(host=row_ptr), ps.DeviceBuffer(host=cnt)
    lib = _native.hip()
    d_lv = ps.DeviceBuffer(64 * 8)
    ps._hip_call(lib.ps_hub_levels(d_ptr.ptr, n, d_cnt.ptr, n, d_lv.ptr, None))
    want = np.bincount(np.floor(np.log2(deg[deg > 0])).astype(int), minlength=32)
    np.testing.assert_array_equal(d_lv.download(np.uint64), np.concatenate([want, want]))
    idx, lst = ps.DeviceBuffer(n * 4), ps.DeviceBuffer(n * 4)
    top = (1 << 63) - 1
    for lo, hi in ((1, top), (64, 4096), (0, top), (top - 1, top)):
        for rows in (True, False):
            v = deg if rows else cnt
            k = ctypes.c_int(-1)
            ps._hip_call(lib.ps_hub_select(d_ptr.ptr if rows else None,
                                           None if rows else d_cnt.ptr, n, lo, hi, idx.ptr,
                                           lst.ptr, ctypes.byref(k), None))
            sel = np.flatnonzero((v >= lo) & (v < hi))
            at = np.full(n, -1, np.int32)
            at[sel] = np.arange(sel.size)
            assert k.value == sel.size
            np.testing.assert_array_equal(idx.download(np.int32), at)
            if sel.size:
                np.testing.assert_array_equal(lst.download(np.int32, sel.size), sel)


@pytest.mark.parametrize("num", [[3, 5], [0, 0, 0, 1], [2, 0, 255, 0, 1], [1, 9, 0, 33, 129, 7]])
def test_tile_list(num):
    # worksets without groups, groups of 32 (no tiles), one tile, several blocks
    setup()
    say(f"hub tiles {num}")
    rng = np.random.default_rng(len(num))
    rows, cols = 300, 500
    hub = np.where(rng.random(rows) < 0.5, 0, -1).astype(np.int32)
    hot = np.where(rng.random(cols) < 0.995, 0, -1).astype(np.int32)
    bufs = [ps.DeviceBuffer(host=a) for a in (hub, hot)]
    hb = _native.HubBlock(rows, cols, rows, cols, bufs[0].ptr, bufs[0].ptr, bufs[1].ptr,
                          bufs[1].ptr, None, None)
    ws = (_native.Workset * len(num))()
    flags, codes = [], []
    for s, g in enumerate(num):
        gs = 32 << max(s - 1, 0)
        c = rng.integers(0, cols, max(g * gs, 1)).astype(np.int32)
        des = rng.integers(0, rows, max(g, 1)).astype(np.int32)
        bufs += [ps.DeviceBuffer(host=c), ps.DeviceBuffer(host=des)]
        ws[s] = _native.Workset(bufs[-2].ptr, None, bufs[-1].ptr, g, 0 if s == 0 else gs, None)
        if s == 0 or gs < 64 or g == 0:
            continue
        f = (hot[c].reshape(-1, 64) >= 0).all(1) & np.repeat(hub[des] >= 0, gs // 64)
        flags.append(f.astype(np.uint8))
        codes.append((s << 27) | np.flatnonzero(f))
    flags = np.concatenate([np.empty(0, np.uint8), *flags])
    codes = np.concatenate([np.empty(0, np.int64), *codes]).astype(np.uint32)
    lib = _native.hip()
    total = lib.ps_hub_tile_total(len(num), ws)
    assert total == flags.size
    d_f, d_c = ps.DeviceBuffer(max(total, 1)), ps.DeviceBuffer(max(total, 1) * 4)
    n = ctypes.c_uint32(77)
    ps._hip_call(lib.ps_hub_tiles(ctypes.byref(hb), len(num), ws, d_f.ptr, d_c.ptr,
                                  ctypes.byref(n), None))
    assert n.value == codes.size
    if total == 0:
        return
    np.testing.assert_array_equal(d_f.download(np.uint8, total), flags)
    if n.value:
        np.testing.assert_array_equal(d_c.download(np.uint32, n.value), codes)
    into = (rng.random(total) < 0.5).astype(np.uint8)
    d_i = ps.DeviceBuffer(host=into)
    ps._hip_call(lib.ps_hub_merge_flags(d_f.ptr, total, d_i.ptr, None))
    np.testing.assert_array_equal(d_i.download(np.uint8), into | flags)
