"""Lakes in every iteration that an outlet reaches (sites of negative area only, no
part of the graph apart): the pipelined iterations look for them, join them and
turn their paths, and none is redone.  Bit for bit against the oracle, on the GPU
and in the CPU emulation."""
import pytest

from test_lasting_lakes import _terrain
from test_sweeps import _check

# (sites of a grid, negative areas, columns apart, slopes, seed)
CASES = [(9, 7, 3, 0, False, 5), (11, 12, 4, 0, True, 8), (30, 20, 8, 0, False, 4), (60, 40, 30, 0, False, 0)]


def _joined(st):
    assert st["iterations"] == st["lake_iterations"] == 40 and st["redone"] == 0
    assert st["host_syncs"] < 3 * st["iterations"]  # (an iteration on its own takes more)


@pytest.mark.parametrize("case", CASES)
def test_emulated_joined_lakes(case):
    from cpu_emu import emu
    from test_cpu_emulation import _emu_solve

    _check(lambda ts: _emu_solve(emu.lib(), ts), [_terrain(*case)])
    st = _emu_solve.last_stats
    _joined({k: getattr(st, k) for k, _ in st._fields_})


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES + [(150, 120, 60, 0, False, 0), (120, 90, 40, 0, True, 0)])
def test_joined_lakes(case):
    from fastlem_amd.device import DeviceTerrain

    def solve(ts):
        t = ts[0]
        d = DeviceTerrain(t["row_ptr"], t["col"], t["length"], t["area"], t["erodibility"], t["uplift"],
                          t["init_elevation"], t["outlets"], t["max_slope"], t["max_iteration"])
        it = d.solve()
        _joined(d.last_stats())
        return [d.elevations()], [it]

    _check(solve, [_terrain(*case)])
