"""Builds next to the end of cpvs_build_noalloc's fixed scratch, where cells, sort arrays and merge tables
take turns in one region.  Words are whole numbers: equality.  Needs a GPU."""
import ctypes as C

import numpy as np
import pytest

import cpvs_amd as cp
from cpvs_amd import _lib

pytestmark = pytest.mark.gpu


def _noalloc(mm, cap):
    out = cp.DeviceArray((cap,), np.uint32, ctx=mm.ctx)
    nw = C.c_uint64()
    _lib.call("cpvs_build_noalloc", mm.ctx.handle, mm.handle, 0, 1, None, out.ptr, cap, C.byref(nw), None)
    words = out.numpy()[:nw.value]
    out.free()
    return words


@pytest.mark.parametrize("merge", ["sort", "table"])
def test_levels_without_leafmasks(merge):
    """Eight ramps over 1024^2, 962,560 nodes at level 0 and a third of that at the next."""
    print("[case] scratch limit", merge, flush=True)
    N = 1024
    x = np.mgrid[0:N, 0:N][1]
    D = (0.1 + 0.68 * ((x * 8 / N) % 1.0)).astype(np.float32)
    c = cp.Context(0)
    try:
        c.set_leafmasks(False)
        mm = cp.MinMaxHierarchy(D, ctx=c)
        assert int(mm.estimate()[0][0]) == 962560
        c.set_merge("table" if merge == "sort" else "sort")
        cs = cp.CompressedShadow.create(mm)
        ref = cs.getDAG()
        cs.close()
        c.set_merge(merge)
        for _ in range(2):
            assert np.array_equal(_noalloc(mm, len(ref)), ref)
    finally:
        c.close()
