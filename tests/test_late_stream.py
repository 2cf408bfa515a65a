"""Work enqueued on a stream may run as late as when the host waits for it: what an
iteration in flight reads from host memory is still there then.  In a CPU emulation
whose streams run at the last moment; unions whose terrains stop at their own
max_iteration, one after the other, bit for bit against the oracle."""
import numpy as np
import pytest

from test_cpu_emulation import _emu_solve
from test_lasting_lakes import _terrain
from test_sweeps import _check


def _lib():
    from cpu_emu import variants

    return variants.lib("late", FLEMU_LATE=1)


def _union(count, lakes, slopes, seed):
    rng = np.random.default_rng([count, lakes, seed])
    ts = [_terrain(int(rng.integers(4, 16)), int(rng.integers(4, 12)), lakes, 0, slopes, seed + i) for i in range(count)]
    for t, cap in zip(ts, rng.permutation(np.arange(4, 4 + count))):
        t["max_iteration"] = int(cap)
    return ts


@pytest.mark.parametrize("lakes", [0, 2])
@pytest.mark.parametrize("pipelining", [1, 2, 3])
def test_terrains_that_stop_one_after_the_other(lakes, pipelining):
    for seed in range(4):
        _check(lambda ts: _emu_solve(_lib(), ts, pipelining=pipelining, compact=(None, 1)[seed % 2]),
               _union(6, lakes, seed == 3, seed))


@pytest.mark.gpu
def test_on_several_streams():
    """Three contexts at a time, whose iterations wait for each other's."""
    import ctypes
    import threading

    from fastlem_amd import _native
    from fastlem_amd.device import batch_descs
    from test_sweeps import _reference

    L = _native.lib()
    unions = [_union(6, 2, False, s) for s in range(12)]
    refs = [[_reference(t) for t in u] for u in unions]
    wrong = []

    def work(k):
        ctx = ctypes.c_void_p()
        _native.check(L.fl_ctx_create(0, ctypes.byref(ctx)))
        for q in np.random.default_rng(k).permutation(np.repeat(np.arange(len(unions)), 8)):
            keep, b, its = [], ctypes.c_void_p(), np.zeros(6, np.uint32)
            descs = batch_descs(unions[q], keep)
            _native.check(L.fl_batch_create(ctx, descs, 6, ctypes.byref(b)))
            _native.check(L.fl_batch_solve(ctx, b, _native.ptr(its, ctypes.c_uint32)))
            for i, (ref, it) in enumerate(refs[q]):
                out = np.empty(len(ref))
                _native.check(L.fl_batch_download(ctx, b, i, _native.ptr(out, ctypes.c_double)))
                if its[i] != it or not np.array_equal(out.view(np.uint64), ref.view(np.uint64)):
                    wrong.append((k, int(q), i, int(its[i]), it))
            L.fl_terrain_destroy(b)
        L.fl_ctx_destroy(ctx)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:5]
