"""Calls on one thread while another thread captures a graph on a stream of its own: the buffer cache's wait
for the device must not invalidate the capture, as hipDeviceSynchronize does.  Needs a GPU."""
import ctypes as C
import threading

import numpy as np
import pytest

import cpvs_amd as cp
import oracle as O

pytestmark = pytest.mark.gpu
THREAD_LOCAL = 1  # hipStreamCaptureModeThreadLocal, as a batch's lanes capture


def test_reused_buffers_leave_a_capture_alone():
    print("[case] buffers reused beside a capture", flush=True)
    hip = C.CDLL("libamdhip64.so")
    c = cp.Context(0)
    other = cp.Context(0)  # its stream is captured
    try:
        N = 8192
        img = cp.gen_depth(N, 0x43505653 + 5, 512, True, ctx=c)
        small = cp.DeviceArray((64,), np.uint32, ctx=other)
        two = [cp.MinMaxHierarchy(img, ctx=c) for _ in range(2)]
        want = two[0].getLevel(5)
        for mm in two:
            mm.close()  # 256 MiB of depth and its levels each: enough pending for the cache to wait
        begun, done, rc = threading.Event(), threading.Event(), {}

        def capture():
            rc["begin"] = hip.hipStreamBeginCapture(other.stream, THREAD_LOCAL)
            begun.set()
            done.wait(60)
            rc["copy"] = hip.hipMemcpyAsync(small.ptr, C.c_void_p(small.ptr.value + 128), C.c_size_t(128), 3, other.stream)
            g = C.c_void_p()
            rc["end"] = hip.hipStreamEndCapture(other.stream, C.byref(g))
            if g:
                hip.hipGraphDestroy(g)
            hip.hipGetLastError()

        t = threading.Thread(target=capture)
        t.start()
        try:
            assert begun.wait(60)
            mm = cp.MinMaxHierarchy(img, ctx=c)  # takes the freed buffers, which needs the device idle
        finally:
            done.set()
            t.join(60)
        assert np.array_equal(mm.getLevel(5), want)
        mm.close()
        assert rc == {"begin": 0, "copy": 0, "end": 0}
    finally:
        c.close()
        other.close()
