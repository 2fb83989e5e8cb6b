"""Graph captures beside other work.  A device synchronisation on any thread invalidates every capture of the
process, and fails itself without waiting: a batch's lanes must get by without their graph, and the
buffer cache must not take the failed wait for done.  Needs a GPU."""
import ctypes as C
import threading

import numpy as np
import pytest

import cpvs_amd as cp

pytestmark = pytest.mark.gpu
SEED0 = 0x43505653
THREAD_LOCAL = 1  # hipStreamCaptureModeThreadLocal, as a batch's lanes capture


@pytest.mark.parametrize("lanes", [1, 4])
def test_graph_forests_beside_device_synchronisations(lanes):
    print("[case] graph forests beside synchronisations", lanes, flush=True)
    hip = C.CDLL("libamdhip64.so")
    c = cp.Context(0)
    try:
        maps = [cp.gen_depth(N, SEED0 + 400 + i, max(1, 32 * N * N >> 20), True, ctx=c)
                for i, N in enumerate([256, 512, 1024] * 4)]
        plain = []
        for d in maps:
            cs = cp.CompressedShadow.create(cp.MinMaxHierarchy(d, ctx=c))
            plain.append(cs.getDAG())
            cs.close()
        stop = threading.Event()

        def sync():
            while not stop.is_set():
                hip.hipDeviceSynchronize()

        t = threading.Thread(target=sync)
        t.start()
        built = []
        try:
            for _ in range(6):
                built.append(cp.build_batch(maps, ctx=c,
                                            config=cp.batch_config(lanes=lanes, forest_mtexels=1, graph=True))[0])
        finally:
            stop.set()
            t.join(60)
        for shadows in built:
            for w, sh in zip(plain, shadows):
                assert np.array_equal(sh.getDAG(), w)
    finally:
        c.close()


def test_reused_buffers_wait_beside_a_capture():
    """Lookups on a stream of their own read a container that is destroyed; the next pyramid's depth is
    copied to a buffer of its size while a third stream, not the library's, is being captured."""
    print("[case] buffers reused beside a capture", flush=True)
    hip = C.CDLL("libamdhip64.so")
    c, reader = cp.Context(0), cp.Context(0)  # (a stream each)
    try:
        big = cp.gen_depth(8192, SEED0 + 5, 512, True, ctx=c)
        img = cp.gen_depth(2048, SEED0 + 6, 128, True, ctx=c)
        q = cp.gen_queries_uniform(SEED0 + 7, 1 << 20, 4, ctx=c)
        mm = cp.MinMaxHierarchy(big, borrow=True, ctx=c)
        k = cp.CompressedShadowContainer(cp.CompressedShadow.create(mm))
        k.setFilterSize(64)
        k.copyToGPU()
        vis = [cp.DeviceArray((1 << 20,), np.float32, ctx=c) for _ in range(2)]
        k.evaluate_pcf(q, None, vis[0])
        c.synchronize()
        want = vis[0].numpy()
        fill = cp.MinMaxHierarchy(cp.gen_depth(4096, SEED0 + 8, 512, True, ctx=c), ctx=c)
        c.release_scratch()  # nothing ready: the next depth takes a pending buffer or new memory
        fill.close()  # more than 64 MiB pending
        begun, done, rc = threading.Event(), threading.Event(), {}

        def capture():
            s = C.c_void_p()
            rc["create"] = hip.hipStreamCreateWithFlags(C.byref(s), 1)
            rc["begin"] = hip.hipStreamBeginCapture(s, THREAD_LOCAL)
            begun.set()
            done.wait(60)
            g = C.c_void_p()
            hip.hipStreamEndCapture(s, C.byref(g))  # (invalid by then, and the stream with it)
            if g:
                hip.hipGraphDestroy(g)
            hip.hipStreamDestroy(s)
            hip.hipGetLastError()

        t = threading.Thread(target=capture)
        t.start()
        try:
            assert begun.wait(60)
            for _ in range(20):
                k.evaluate_pcf(q, None, vis[1], stream=reader.stream)
            k.close()
            one = cp.MinMaxHierarchy(img, ctx=c)  # 16 MiB, the container's words' and links' sizes
        finally:
            done.set()
            t.join(60)
        reader.synchronize()
        assert rc == {"create": 0, "begin": 0}
        assert np.array_equal(vis[1].numpy(), want)
        assert np.array_equal(one.getLevel(0), img.numpy())
    finally:
        for x in (c, reader):
            x.close()
