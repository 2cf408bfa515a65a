"""Long chains, whose tiles guess their values from exact sums and check the
guess: areas on coarse grids (terms halfway between two values, of either
parity), on one binade and over many, ones that no guess fits (zero, negative,
huge), tiles around the length from which they guess, and positions with as
many light children as a list holds and more, on either side of the heavy
child.  Bit for bit against the oracle, on the GPU and in the CPU emulation."""
import numpy as np
import pytest

from test_sweeps import _check, _terrain

AREAS = ("grid", "coarse", "equal", "wide", "odd")


def _chain(spine, leaves, first, slopes, areas):
    t = _terrain(spine, leaves, first, slopes)
    n = len(t["area"])
    rng = np.random.default_rng([spine, leaves, AREAS.index(areas)])
    t["area"] = {"grid": rng.integers(1, 1 << 12, n) / 1024.0,
                 "coarse": rng.integers(1, 1 << 20, n) * (2.0 ** -20 + 2.0 ** -52),
                 "equal": np.full(n, 1.0 / 3.0),
                 "wide": 2.0 ** rng.uniform(-40, 12, n),
                 "odd": np.where(rng.random(n) < 0.02, rng.choice([0.0, -0.5, 1e300, 1e-300], n), rng.uniform(0.5, 2.0, n)),
                 }[areas]
    t["max_iteration"] = 3
    return t


@pytest.mark.parametrize("spine,leaves,first,slopes,areas", [
    (400, 1, False, False, "grid"), (300, 3, True, True, "coarse"), (177, 8, False, False, "equal"),
    (60, 8, True, False, "wide"), (40, 9, True, False, "wide"), (129, 9, False, True, "odd")])
def test_emulated_long_chains(spine, leaves, first, slopes, areas):
    from cpu_emu import emu
    from test_cpu_emulation import _emu_solve

    _check(lambda ts: _emu_solve(emu.lib(), ts), [_chain(spine, leaves, first, slopes, areas)])


@pytest.mark.gpu
@pytest.mark.parametrize("areas", AREAS)
@pytest.mark.parametrize("leaves,first,slopes", [(0, False, False), (1, False, True), (3, True, False), (5, False, False),
                                                 (8, False, False), (8, True, True), (9, False, False), (9, True, False)])
def test_long_chains(leaves, first, slopes, areas):
    from fastlem_amd.device import DeviceBatch

    def solve(ts):
        b = DeviceBatch(ts)
        its = b.solve()
        return [b.elevations(i) for i in range(len(ts))], its

    spines = (128, 130, 176, 177, 178, 255, 256, 257, 1000, 1025, 3000)
    _check(solve, [_chain(s, leaves, first, slopes, areas) for s in spines])
    _check(solve, [_chain(2049, leaves, first, slopes, areas)])
