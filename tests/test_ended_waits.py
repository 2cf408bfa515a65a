"""Sweeps whose waits end without their values: the iteration is redone behind
barriers, the ones after it are pipelined again (once more the next time, then
after twice as many iterations), and a later solve of the same terrain starts
afresh.  In a CPU emulation where a wait of the one-launch sweeps ends at its
first poll, so that nearly every such launch has one; bit for bit against the
oracle."""
import ctypes

import numpy as np
import pytest

from test_cpu_emulation import _emu_solve
from test_lasting_lakes import _terrain as lakes
from test_long_chains import _chain
from test_start_order import _strip
from test_sweeps import _check, _reference


def _ended():
    from cpu_emu import variants

    return variants.lib("ended_waits", FL_SPIN_FOLD=1)


def _descs(t):
    from fastlem_amd.device import batch_descs

    keep = []
    return batch_descs([t], keep), keep


CASES = {
    "chain": lambda: _chain(1300, 2, False, False, "grid"),
    "chain with slopes": lambda: _chain(500, 9, True, True, "coarse"),
    "strip": lambda: _strip(False),
    "strip with slopes": lambda: _strip(True),
    "lakes": lambda: lakes(60, 50, 6, 2, False, 5),
}


@pytest.mark.parametrize("case", CASES)
def test_solved_again(case):
    from cpu_emu import emu
    from fastlem_amd import _native

    L, t = _ended(), CASES[case]()
    t["max_iteration"] = 12
    ref, rit = _reference(t)
    ctx, d = ctypes.c_void_p(), ctypes.c_void_p()
    emu.check(L, L.fl_ctx_create(0, ctypes.byref(ctx)))
    redone = []
    try:
        descs, keep = _descs(t)
        emu.check(L, L.fl_terrain_create(ctx, descs, ctypes.byref(d)))
        for _ in range(3):
            it = ctypes.c_uint32()
            emu.check(L, L.fl_terrain_solve(ctx, d, t["max_iteration"], ctypes.byref(it)))
            out, st = np.empty(len(ref)), _native.SolveStats()
            emu.check(L, L.fl_terrain_download(ctx, d, _native.ptr(out, ctypes.c_double)))
            emu.check(L, L.fl_terrain_last_stats(d, ctypes.byref(st)))
            assert it.value == rit and np.array_equal(out.view(np.uint64), ref.view(np.uint64))
            redone.append(st.redone)
        L.fl_terrain_destroy(d)
    finally:
        L.fl_ctx_destroy(ctx)
    assert min(redone) > 0, redone  # pipelined iterations were tried, and redone


def test_unions():
    _check(lambda ts: _emu_solve(_ended(), ts),
           [_chain(300, 3, False, False, "odd"), lakes(40, 30, 0, 3, False, 6), _chain(260, 1, False, False, "wide")])
    assert _emu_solve.last_stats.redone > 0
    # (terrains that stop early leave the union)
    _check(lambda ts: _emu_solve(_ended(), ts, compact=1),
           [_chain(200, 1, False, False, "equal"), lakes(30, 30, 3, 2, False, 7), lakes(9, 9, 0, 0, False, 8)])
