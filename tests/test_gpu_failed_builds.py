"""A build that fails returns with nothing of it left on the GPU: its scratch is the context's, or for
cpvs_build_noalloc the device's, and the next call may come on another stream.  Needs a GPU."""
import ctypes as C

import numpy as np
import pytest

import cpvs_amd as cp
from cpvs_amd import _lib
import oracle as O

pytestmark = pytest.mark.gpu
SEED0 = 0x43505653


def _say(*a):
    print("[case]", *a, flush=True)


def _noalloc(mm, out, cap):
    nw = C.c_uint64()
    _lib.call("cpvs_build_noalloc", mm.ctx.handle, mm.handle, 0, 1, None, out.ptr, cap, C.byref(nw), None)
    return out.numpy()[:nw.value]


def test_refused_output_then_build_on_another_stream():
    """An output one word short is refused after the last merge launch was queued; the next build lays
    out the same fixed scratch on another context's stream at once."""
    a, b = cp.Context(0), cp.Context(0)
    try:
        Da, Db = O.gen_depth(1024, SEED0 + 61, 32, True), O.gen_depth(512, SEED0 + 62, 16, True)
        ma, mb = cp.MinMaxHierarchy(Da, ctx=a), cp.MinMaxHierarchy(Db, ctx=b)
        ref_a, ref_b = (cp.CompressedShadow.create(m).getDAG() for m in (ma, mb))
        out_a, out_b = cp.DeviceArray((len(ref_a),), np.uint32, ctx=a), cp.DeviceArray((len(ref_b),), np.uint32, ctx=b)
        for k in range(8):
            _say("refused output, then another stream", k)
            with pytest.raises(cp.CpvsError) as e:
                _noalloc(ma, out_a, len(ref_a) - 1)
            assert e.value.code == _lib.CPVS_EINVAL
            assert np.array_equal(_noalloc(mb, out_b, len(ref_b)), ref_b)
            assert np.array_equal(_noalloc(ma, out_a, len(ref_a)), ref_a)
    finally:
        a.close()
        b.close()


def test_refused_scratch_then_build_on_another_stream():
    """A map that needs more than the fixed scratch is refused right after its counts."""
    a, b = cp.Context(0), cp.Context(0)
    try:
        big = cp.MinMaxHierarchy(np.random.default_rng(3).random((2048, 2048), dtype=np.float32), ctx=a)
        mb = cp.MinMaxHierarchy(O.gen_depth(512, SEED0 + 62, 16, True), ctx=b)
        ref = cp.CompressedShadow.create(mb).getDAG()
        out_a, out_b = cp.DeviceArray((1,), np.uint32, ctx=a), cp.DeviceArray((len(ref),), np.uint32, ctx=b)
        for k in range(4):
            _say("refused scratch, then another stream", k)
            with pytest.raises(cp.CpvsError) as e:
                _noalloc(big, out_a, 1)
            assert e.value.code == _lib.CPVS_EINVAL and "scratch" in str(e.value)
            assert np.array_equal(_noalloc(mb, out_b, len(ref)), ref)
    finally:
        a.close()
        b.close()
