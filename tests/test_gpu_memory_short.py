"""An allocation that fails is tried again without the cache of freed buffers, so maps, containers and
DAGs that a program destroyed do not count against it.  Needs a GPU."""
import numpy as np
import pytest

import cpvs_amd as cp
import oracle as O

pytestmark = pytest.mark.gpu


def test_a_failing_allocation_empties_the_cache():
    print("[case] allocation beyond the device", flush=True)
    c = cp.Context(0)
    try:
        srv = cp.Server(serial=True, ctx=c)  # (its statistics report the cache)
        mm = cp.MinMaxHierarchy(O.gen_depth(512, 0x43505653, 16, True), ctx=c)  # a copied depth map
        k = cp.CompressedShadowContainer(cp.CompressedShadow.create(mm))
        k.copyToGPU()
        mm.close()
        k.close()
        assert srv.stats()["cached_bytes"] >= 4 * 512 * 512
        with pytest.raises(cp.CpvsError) as e:
            cp.DeviceArray((1 << 46,), np.uint8, ctx=c)  # no device holds 64 TiB
        assert e.value.code == 2  # CPVS_ENOMEM
        assert srv.stats()["cached_bytes"] == 0
        mm = cp.MinMaxHierarchy(O.gen_depth(64, 0x43505653, 2, True), ctx=c)  # and the context goes on
        assert cp.CompressedShadow.create(mm).num_words() > 0
        srv.close()
    finally:
        c.close()
