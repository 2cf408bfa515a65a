"""A pipelined iteration whose result is not used (the solve's last one was before
it) may have ended a wait without its value like any other: the hand-over words
that it left do not reach the next solve.  In a CPU emulation where the waits of
chosen launches end at their first poll; bit for bit against the oracle."""
import ctypes

import numpy as np
import pytest

from test_lasting_lakes import _terrain
from test_sweeps import _reference


class _Polls:
    """The library with the number of sweep launches and those whose waits are short."""

    def __init__(self):
        from cpu_emu import variants

        self.lib = variants.lib("polls", source="polls.cpp", header="polls.h", FL_SPIN_FOLD="flemu_polls()")
        self._at = lambda name: ctypes.c_uint32.in_dll(self.lib, name)

    def start(self, first=0xFFFFFFFF, end=0xFFFFFFFF):
        for name, v in (("flemu_launches", 0), ("flemu_short_from", first), ("flemu_short_to", end)):
            self._at(name).value = v

    def launches(self):
        return self._at("flemu_launches").value


@pytest.mark.parametrize("nx,ny,seed", [(16, 12, 5), (16, 12, 17), (16, 12, 29), (40, 20, 86)])
def test_after_the_last_iteration(nx, ny, seed):
    """Every basin recomputed in every iteration: the one in flight when the solve
    ends has the whole terrain's sweeps."""
    from cpu_emu import emu
    from fastlem_amd import _native
    from fastlem_amd.device import batch_descs

    P = _Polls()
    L = P.lib
    t = _terrain(nx, ny, 0, 0, False, seed)
    t["max_iteration"] = 200
    ref, rit = _reference(t)
    assert rit < 200
    keep = []
    descs = batch_descs([t], keep)
    ctx, d = ctypes.c_void_p(), ctypes.c_void_p()
    emu.check(L, L.fl_ctx_create(0, ctypes.byref(ctx)))

    def solve(*short):
        P.start(*short)
        it, out, st = ctypes.c_uint32(), np.empty(len(ref)), _native.SolveStats()
        emu.check(L, L.fl_terrain_solve(ctx, d, 200, ctypes.byref(it)))
        emu.check(L, L.fl_terrain_download(ctx, d, _native.ptr(out, ctypes.c_double)))
        emu.check(L, L.fl_terrain_last_stats(d, ctypes.byref(st)))
        assert it.value == rit and np.array_equal(out.view(np.uint64), ref.view(np.uint64))
        return st.redone

    try:
        emu.check(L, L.fl_ctx_set_recompute_all(ctx, 1))
        emu.check(L, L.fl_terrain_create(ctx, descs, ctypes.byref(d)))
        redone = solve()
        last = P.launches() - 2  # the last iteration's two sweeps
        assert solve(last, last + 2) == redone  # (not looked at: the solve was over)
        assert solve() == redone
        L.fl_terrain_destroy(d)
    finally:
        L.fl_ctx_destroy(ctx)
