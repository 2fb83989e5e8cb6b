"""The scratch that a build lays out, from its node counts (CPU only: sizes, no compute call).  The
function is the library's own, which builds, admission and estimates share."""
import ctypes as C

import pytest

from cpvs_amd import _lib

LEVELS = 24


def scratch_bytes(cnt, R, leaf, ncol=0, col_list=False, table=True, small=True):
    f = C.CDLL(_lib.LIB_PATH)._ZN4cpvs19build_scratch_bytesEPKmibjbbb
    f.restype = C.c_size_t
    f.argtypes = [C.POINTER(C.c_uint64), C.c_int, C.c_bool, C.c_uint32, C.c_bool, C.c_bool, C.c_bool]
    return f((C.c_uint64 * LEVELS)(*cnt), R, leaf, ncol, col_list, table, small)


def counts(bottom, R, deepest, ratio):
    """Nodes per level: `deepest` at the bottom, `ratio` times fewer at each level above."""
    c = [0] * LEVELS
    for L in range(bottom, R + 1):
        c[L] = max(1, int(deepest / ratio ** (L - bottom)))
    c[R] = 1
    return c


@pytest.mark.parametrize("table,per_node", [(True, 89), (False, 109)], ids=["table", "sort"])
def test_counts_beyond_32_bits(table, per_node):
    """An estimate for more than 2^32 nodes at a level grows with them: a leaf node takes its mask,
    identity, unique entry and offset (16 bytes), flag (1), leafmask row (64), run head and column entry
    (8), and in a sort its keys, values, their copies and its segment (20)."""
    need = []
    for nodes in ((1 << 32) - 16, 1 << 34):
        c = counts(2, 15, 1000, 2)
        c[2] = nodes
        need.append(scratch_bytes(c, 15, True, 8192 * 8192, table=table, small=False))
    assert need[1] - need[0] >= per_node * ((1 << 34) - (1 << 32))


# Counts whose builds fitted the fixed scratch when one table, of the largest level's size, and one set of
# sort arrays served all levels: without leafmasks, halving and quartering levels, next to its end.
FITTING = [
    ([794417, 411119, 212758, 110104, 56980, 29487, 15260, 1], False),
    ([747276, 386278, 199672, 103213, 53352, 27578, 14255, 1], True),
    ([962560, 329728, 93184, 25000, 6600, 1800, 450, 60, 1], False),
    ([962560, 329728, 93184, 25000, 6600, 1800, 450, 60, 1], True),
]


@pytest.mark.parametrize("cnt,table", FITTING, ids=lambda v: str(v[0]) if isinstance(v, list) else ("table" if v else "sort"))
def test_fixed_scratch_takes_what_it_took(cnt, table):
    limit = C.CDLL(_lib.LIB_PATH).cpvs_build_noalloc_scratch_bytes
    limit.restype = C.c_size_t
    c = cnt + [0] * (LEVELS - len(cnt))
    for small in (True, False):
        assert scratch_bytes(c, len(cnt) - 1, False, table=table, small=small) <= limit()
