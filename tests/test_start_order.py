"""The sweeps wait for nothing that has not started: in a CPU emulation that runs
a launch's workgroups one after the other, each to its end, the last one first, no
wait ends without its value.  Bit for bit against the oracle, and with as many
host synchronisations as in the usual order (an ended wait takes more)."""
import numpy as np
import pytest

from test_cpu_emulation import _emu_solve
from test_lasting_lakes import _terrain as lakes
from test_long_chains import _chain
from test_sweeps import _check


def _strip(slopes):
    from fastlem_amd.device import DeviceBatch
    from fastlem_amd.workloads import config_strip

    t = DeviceBatch.terrain_of(config_strip(256, 12))
    t["max_slope"] = np.full(len(t["area"]), 0.4) if slopes else None
    t["max_iteration"] = 12
    return t


CASES = {
    "strip": lambda: [_strip(False)],
    "strip with slopes": lambda: [_strip(True)],
    "union": lambda: [_chain(1300, 2, False, False, "grid"), lakes(60, 50, 0, 2, False, 3), _chain(40, 9, True, False, "wide")],
    "union with slopes": lambda: [_chain(700, 3, True, True, "odd"), lakes(40, 40, 3, 0, True, 4)],
}


@pytest.mark.parametrize("case", CASES)
def test_last_workgroup_first(case):
    from cpu_emu import emu, variants

    syncs = []

    def solve(L):
        def run(ts):
            r = _emu_solve(L, ts)
            syncs.append((_emu_solve.last_stats.host_syncs, _emu_solve.last_stats.redone))
            return r
        return run

    ts = CASES[case]()
    _check(solve(emu.lib()), ts)
    _check(solve(variants.lib("last_first", FLEMU_LAST_FIRST=1, FL_SPIN_FOLD=512)), ts)
    assert syncs[0] == syncs[1]
