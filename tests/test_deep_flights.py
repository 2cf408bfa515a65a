"""Pipelined iterations whose decomposition is deeper than their placement takes:
they and the ones behind them do nothing and are redone; after one near the limit
the bucket offsets are scanned in a launch of their own.  In CPU emulations that
take two and three rounds (64 otherwise), with lakes that last, alone and in
unions; bit for bit against the oracle."""
import pytest

from test_cpu_emulation import _emu_solve
from test_lasting_lakes import _terrain
from test_sweeps import _check

# (sites of a grid, negative areas, columns apart, slopes, seed)
CASES = [(30, 8, 6, 2, True, 42), (30, 8, 6, 2, True, 52), (25, 25, 8, 3, False, 48), (16, 12, 4, 0, False, 31),
         (14, 5, 2, 0, False, 54)]


def _solve(rounds, ts, **kw):
    from cpu_emu import emu, variants

    L = variants.lib(f"scan{rounds}", FL_SCAN_ROUNDS=rounds) if rounds else emu.lib()
    _check(lambda x: _emu_solve(L, x, **kw), ts)
    return _emu_solve.last_stats


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("pipelining", [1, 3])  # (3: replayed graphs)
def test_deeper_than_the_limit(case, pipelining):
    ts = [_terrain(*case)]
    usual, st = _solve(0, ts, pipelining=pipelining), _solve(3, ts, pipelining=pipelining)
    assert st.max_sweep_rounds > 3 and usual.redone < st.redone < st.iterations


def test_scanned_in_a_launch():
    for case in CASES:
        st = _solve(2, [_terrain(*case)])
        assert st.max_sweep_rounds > 2 and st.redone < st.iterations


@pytest.mark.parametrize("rounds", [2, 3])
def test_unions(rounds):
    _solve(rounds, [_terrain(*c) for c in CASES if not c[4]])
    _solve(rounds, [_terrain(*c) for c in CASES], compact=1, recompute_all=1)
