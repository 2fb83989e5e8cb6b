"""Merge tables of all levels are emptied as one run, which may hold more than 2^32 slots.  Needs a GPU."""
import ctypes as C

import numpy as np
import pytest

import cpvs_amd as cp
from cpvs_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", [1, 255, 256, 257, 65536 * 256 + 1, (1 << 32) + 513])
def test_table_clear(slots):
    print("[case] table clear", slots, flush=True)
    clear = C.CDLL(_lib.LIB_PATH)._ZN4cpvs11table_clearEPmmP12ihipStream_t
    clear.argtypes = [C.c_void_p, C.c_uint64, C.c_void_p]
    c = cp.Context(0)
    try:
        guard = 64
        buf = cp.DeviceArray((slots + guard,), np.uint64, ctx=c)
        # the first and the last slots, those around 2^32, and the words behind the tables
        at = sorted({a for a in [0, *range(slots - 600, slots + guard), *range((1 << 32) - 300, (1 << 32) + 300)]
                     if 0 <= a < slots + guard})
        runs = np.split(np.array(at), np.flatnonzero(np.diff(at) != 1) + 1)
        for r in runs:
            z = np.zeros(len(r), np.uint64)
            _lib.call("cpvs_memcpy_h2d", c.handle, C.c_void_p(buf.ptr.value + 8 * int(r[0])),
                      z.ctypes.data_as(C.c_void_p), z.nbytes)
        clear(buf.ptr, slots, c.stream)
        for r in runs:
            z = np.zeros(len(r), np.uint64)
            _lib.call("cpvs_memcpy_d2h", c.handle, z.ctypes.data_as(C.c_void_p),
                      C.c_void_p(buf.ptr.value + 8 * int(r[0])), z.nbytes)
            want = np.where(r < slots, np.uint64(0xFFFFFFFFFFFFFFFF), np.uint64(0))
            assert np.array_equal(z, want), (int(r[0]), len(r))
        buf.free()
    finally:
        c.close()
