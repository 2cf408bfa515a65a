"""The sweeps at the sizes where their tiles, lists and hand-overs change
form: chains around the short / long cutoff and around one and several tiles,
sites with as many light children as a list holds and more, before the heavy
child and after it, with and without max slopes.  Bit for bit against the
oracle, on the GPU and in the CPU emulation."""
import numpy as np
import pytest

from conftest import comb_terrain

SLOPES = (0.3, 0.0, np.nan, 1.2, 1e-300, np.pi / 2, 0.05)  # tan: ordinary, zero, none, tiny, huge


def _terrain(spine, leaves, leaves_first, slopes):
    """A comb (one heavy chain of `spine` sites with `leaves` light children
    each), its rows reversed when the light children are to be folded before
    the heavy one."""
    t = comb_terrain(spine=spine, leaves=leaves, seed=spine + leaves)
    if leaves_first:
        rp = t["row_ptr"].astype(np.int64)
        back = np.concatenate([np.arange(rp[i + 1] - 1, rp[i] - 1, -1) for i in range(len(rp) - 1)])
        t["col"], t["length"] = t["col"][back], t["length"][back]
    rng = np.random.default_rng(spine)
    n = len(t["area"])
    t["erodibility"], t["uplift"] = rng.uniform(0.2, 5.0, n), rng.uniform(0.0, 2.0, n)
    t["max_slope"] = np.resize(np.array(SLOPES), n) if slopes else None
    t["max_iteration"] = 6
    return t


def _reference(t):
    from oracle import flo

    g = flo.Graph(t["row_ptr"], t["col"], t["length"])
    h, it, _ = flo.generate(g, t["area"], t["erodibility"], t["uplift"], t["init_elevation"], t["outlets"],
                            max_iteration=t["max_iteration"], max_slope=t["max_slope"])
    return h, it


def _check(solve, terrains):
    outs, its = solve(terrains)
    for t, out, it in zip(terrains, outs, its):
        ref, rit = _reference(t)
        assert it == rit
        assert np.array_equal(out.view(np.uint64), ref.view(np.uint64))


@pytest.mark.parametrize("slopes", [False, True])
@pytest.mark.parametrize("spine,leaves,first", [(2, 1, False), (16, 4, False), (17, 7, True), (129, 5, True)])
def test_emulated_sweeps(spine, leaves, first, slopes):
    from cpu_emu import emu
    from test_cpu_emulation import _emu_solve

    _check(lambda ts: _emu_solve(emu.lib(), ts), [_terrain(spine, leaves, first, slopes)])


@pytest.mark.gpu
@pytest.mark.parametrize("slopes", [False, True])
@pytest.mark.parametrize("first", [False, True])
@pytest.mark.parametrize("leaves", [1, 4, 5, 6, 7])
def test_sweeps(leaves, first, slopes):
    """Spines of every length at an edge, alone and as one union."""
    from fastlem_amd.device import DeviceBatch

    def solve(ts):
        b = DeviceBatch(ts)
        its = b.solve()
        return [b.elevations(i) for i in range(len(ts))], its

    ts = [_terrain(s, leaves, first, slopes) for s in (1, 2, 15, 16, 17, 33, 64, 65, 127, 128, 129, 256, 257, 513)]
    _check(solve, ts)
    for t in ts:
        _check(solve, [t])
