"""Key collisions in levels small enough for the one-workgroup insert, whose compares run beside the write
of the words only.  With the inner key hashes cut to a few bits, distinct subtrees share slots; the
compares must catch it and send the build down the sort path, whose words equal the oracle's.  Needs a
GPU."""
import numpy as np
import pytest

import cpvs_amd as cp
import oracle as O

pytestmark = pytest.mark.gpu
SEED0 = 0x43505653


@pytest.mark.parametrize("N,bits", [(64, 1), (64, 2), (128, 2), (128, 8), (256, 2), (256, 8)])
def test_small_levels_detect_collisions(N, bits):
    """White noise: nearly all subtrees are distinct, and level 3 of 256^2 holds 16^3 = 4096 nodes."""
    print("[case] small collisions", N, bits, flush=True)
    D = np.random.default_rng(SEED0 + N).random((N, N), dtype=np.float32)
    words, n = O.create(O.Pyramid(D), 0, 1, merge_mode=1)
    c = cp.Context(0)
    try:
        mm = cp.MinMaxHierarchy(D, ctx=c)
        cs = cp.CompressedShadow.create(mm)
        assert cs.merge_info()[0] == "table"
        nodes, uniq = cs.level_stats()
        assert nodes[3:].max() <= 4096  # every inner level takes the one-workgroup insert
        assert uniq[3:].max() > 2 ** bits  # more distinct keys than cut hashes
        assert np.array_equal(cs.getDAG(), words)
        c.set_hash_bits(0, bits)
        cs = cp.CompressedShadow.create(mm)
        assert cs.merge_info()[0] == "sort"
        assert np.array_equal(cs.getDAG(), words)
    finally:
        c.close()
