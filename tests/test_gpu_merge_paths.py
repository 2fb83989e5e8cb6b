"""The merge's dispatch by size: where the key compares run (with the insert or beside the write of the
words), how the tiles' totals are scanned, one or two nodes a thread.  The table merge's words equal
the sort merge's, which the oracle tests pin, at sizes on both sides of each line, and key collisions
are caught on both sides.  Words are whole numbers: equality.  Needs a GPU."""
import numpy as np
import pytest

import cpvs_amd as cp

pytestmark = pytest.mark.gpu
SEED0 = 0x43505653


def _say(*a):
    print("[case]", *a, flush=True)


def _words(c, N, T=1, t=0, boxes=None):
    D = cp.gen_depth(N, SEED0 + N, boxes if boxes is not None else max(1, 32 * N * N // (1 << 20)), True, ctx=c)
    mm = cp.MinMaxHierarchy(D, ctx=c)
    cs = cp.CompressedShadow.create(mm, t, T)
    w, how = cs.getDAG(), cs.merge_info()[0]
    cs.close()
    mm.close()
    D.free()
    return w, how


@pytest.mark.parametrize("N,T,t", [(16, 1, 0), (32, 1, 0), (64, 2, 1), (512, 1, 0), (1024, 4, 2), (2048, 1, 0), (4096, 1, 0),
                                   (8192, 1, 0), (8192, 8, 4)])
def test_table_words_equal_sort_words(N, T, t):
    _say("merge sizes", N, T, t)
    c = cp.Context(0)
    try:
        a, how = _words(c, N, T, t)
        assert how == "table"
        c.set_merge("sort")
        b, how = _words(c, N, T, t)
        assert how == "sort"
        assert np.array_equal(a, b)
    finally:
        c.close()


@pytest.mark.parametrize("N", [2048, 8192])
@pytest.mark.parametrize("bits", [(2, 0), (18, 0), (0, 2), (0, 18)], ids=lambda b: f"leaf{b[0]}-inner{b[1]}")
def test_collisions_of_large_levels(N, bits):
    """Levels above and below the size from which the inserts compare the keys themselves."""
    _say("large collisions", N, bits)
    c = cp.Context(0)
    try:
        a, how = _words(c, N)
        assert how == "table"
        c.set_hash_bits(*bits)
        b, how = _words(c, N)
        assert how == "sort"
        assert np.array_equal(a, b)
    finally:
        c.close()
