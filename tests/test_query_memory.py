"""A query's device memory goes back: after a query of many points the card has as
much free memory as before it, up to the block that the library keeps for the next
one, while the context and the interpolator live on."""
import ctypes

import numpy as np
import pytest


@pytest.mark.gpu
def test_large_query_gives_its_memory_back():
    from fastlem_amd import _native
    from fastlem_amd.surface import TerrainInterpolator2D

    hip = _native.lib()  # (the HIP runtime's functions, through the library that is linked to it)
    rng = np.random.default_rng(3)
    n, m = 2000, 8_000_000
    interp, z = TerrainInterpolator2D(rng.uniform(0.0, 10.0, n), rng.uniform(0.0, 10.0, n)), rng.uniform(0.0, 1.0, n)

    def query(k):
        v, ok = interp.interpolate_many(z, rng.uniform(0.0, 10.0, k), rng.uniform(0.0, 10.0, k))
        assert np.isfinite(v[ok]).all() and ok.mean() > 0.9
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipDeviceSynchronize() == 0
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    query(1000)  # (the kernel and the first block)
    before = query(1000)
    after = query(m)  # 25 bytes a point: 200 MB
    interp.close()
    assert before - after <= 64 << 20, (before, after)
