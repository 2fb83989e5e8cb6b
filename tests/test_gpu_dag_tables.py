"""The device memory of a DAG's lookup tables: what a DAG that leaves a server gives back.  The sizes are
those of the context's cache of freed buffers, which the server's statistics report.  Needs a GPU."""
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


def _server_dag(srv, ticket):
    h, nw = C.c_void_p(), C.c_uint64()
    _lib.call("cpvs_server_dag", srv.handle, ticket, C.byref(h))
    _lib.call("cpvs_dag_info", h, None, C.byref(nw), None)
    return h, nw.value


@pytest.mark.parametrize("evict", [False, True], ids=["released", "evicted"])
def test_server_dags_give_their_tables_back(evict):
    _say("server tables", evict)
    c = cp.Context(0)
    try:
        depth = cp.DeviceArray.from_numpy(O.gen_depth(512, SEED0 + 81, 16, True), ctx=c)
        probe = cp.Server(serial=True, ctx=c)
        probe.wait(probe.build(depth))
        st = probe.stats()
        mm = cp.MinMaxHierarchy(depth, ctx=c)
        dag_max = mm.estimate()[2]
        mm.close()
        probe.close()
        # the lane's scratch and one build's bound, but not that beside a resident DAG
        budget = st["scratch_bytes"] + dag_max + st["resident_bytes"] // 2 if evict else 1 << 30
        c.release_scratch()
        srv = cp.Server(serial=True, budget_bytes=budget, ctx=c)
        try:
            t = srv.build(depth)
            srv.wait(t)
            h, words = _server_dag(srv, t)
            _lib.call("cpvs_dag_set_top_levels", h, 3)
            _lib.call("cpvs_dag_set_top_levels", h, 4)  # the replaced table is kept until the DAG goes
            before = srv.stats()["cached_bytes"]
            tables = 8 * (8 ** 3 + 8 ** 4) + 8 * words  # two tables and the links
            if evict:
                late = srv.build(depth)
                srv.wait(late)
                assert srv.resident() == [late]
                assert srv.stats()["cached_bytes"] - before >= tables  # (its words serve the second DAG)
            else:
                srv.release(t)
                assert srv.stats()["cached_bytes"] - before >= tables + 4 * words
        finally:
            srv.close()
    finally:
        c.close()


@pytest.mark.parametrize("levels,links", [(5, False), (4, True), (3, True)])
def test_links_only_where_a_walk_reads_them(levels, links):
    """A 256^2 DAG has 5 inner levels above the last: with all of them in the table no walk takes a link,
    with one or two left (and links of less than 2 MiB) it does."""
    _say("links rule", levels)
    c = cp.Context(0)
    try:
        mm = cp.MinMaxHierarchy(O.gen_depth(256, SEED0 + 82, 8, True), ctx=c)
        cs = cp.CompressedShadow.create(mm)
        mm.close()
        words = cs.num_words()
        q = cp.DeviceArray.from_numpy(O.gen_queries_uniform(SEED0 + 83, 4096, 3), ctx=c)
        want = cs.evaluate(q).numpy()
        srv = cp.Server(serial=True, ctx=c)  # (its statistics report the cache)
        c.release_scratch()
        cs.setTopLevels(levels)
        assert cs.top_levels() == levels
        assert np.array_equal(cs.evaluate(q).numpy(), want)
        before = srv.stats()["cached_bytes"]
        cs.close()
        assert srv.stats()["cached_bytes"] - before == 4 * words + 8 * 8 ** levels + (8 * words if links else 0)
        srv.close()
    finally:
        c.close()
