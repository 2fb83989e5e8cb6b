"""Maps large enough for one leaf column per lane (2^15 columns, 2048^2 and up), with non-finite texels, which
leave their columns to the waves, and forests on both sides of the sizes that choose their kernels.
Words are whole numbers: equality.  Needs a GPU."""
import numpy as np
import pytest

import cpvs_amd as cp
import oracle as O
from tests.nanmaps import sparse_nan_map

pytestmark = pytest.mark.gpu
SEED0 = 0x43505653


@pytest.mark.parametrize("T,t", [(1, 0), (2, 1)])
def test_non_finite_columns_in_a_single_build(T, t):
    print("[case] non-finite columns", T, t, flush=True)
    D = sparse_nan_map(2048, SEED0 + 7, 0.0002, 0.0001)
    want, _ = O.create(O.Pyramid(D), t, T, merge_mode=1)
    c = cp.Context(0)
    try:
        cs = cp.CompressedShadow.create(cp.MinMaxHierarchy(D, ctx=c), t, T)
        assert np.array_equal(cs.getDAG(), want)
    finally:
        c.close()


# (sides, leaf nodes of the forest at least, at most): below 2^15 columns; lanes with totals in the offsets
# launch (1024 tiles of 2048 nodes); above both, inner levels beyond 2^18 and 2^20 nodes.
FORESTS = [([256, 512, 512], 0, 1 << 15), ([1024, 1024, 2048, 512], 1 << 17, 1 << 20), ([4096] * 4 + [256], 1 << 22, 1 << 26)]


@pytest.mark.parametrize("sides,least,most", FORESTS, ids=lambda v: "+".join(map(str, v)) if isinstance(v, list) else str(v))
def test_forests_of_every_size_equal_single_builds(sides, least, most):
    print("[case] forest sizes", sides, flush=True)
    c = cp.Context(0)
    try:
        maps = [cp.gen_depth(N, SEED0 + 300 + i, max(1, 32 * N * N >> 20), True, ctx=c) for i, N in enumerate(sides)]
        shadows, _ = cp.build_batch(maps, ctx=c, config=cp.batch_config(lanes=1, forest_mtexels=4096))
        leaves = 0
        for d, sh in zip(maps, shadows):
            one = cp.CompressedShadow.create(cp.MinMaxHierarchy(d, ctx=c))
            leaves += int(one.level_stats()[0][2])
            assert sh.merge_info()[0] == "table"
            assert np.array_equal(sh.getDAG(), one.getDAG())
        print("leaf nodes", leaves, flush=True)
        assert least <= leaves <= most
    finally:
        c.close()
