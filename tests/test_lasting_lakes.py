"""Lakes in every iteration, which pipelined iterations join: sites whose
drainage area gives no response time (negative areas), and a part of the graph
that no outlet reaches.  Bit for bit against the oracle, alone and in unions, on
the GPU and in the CPU emulation."""
import numpy as np
import pytest

from test_sweeps import _check


def _terrain(nx, ny, negative, apart, slopes, seed):
    """A jittered grid with its rim's west side as outlets; `negative` sites of
    negative area; the last `apart` columns not connected to the others."""
    rng = np.random.default_rng([nx, ny, seed])
    n = nx * ny
    x, y = np.tile(np.arange(nx), ny) + rng.uniform(-0.3, 0.3, n), np.repeat(np.arange(ny), nx) + rng.uniform(-0.3, 0.3, n)
    rows = [[] for _ in range(n)]
    for j in range(ny):
        for i in range(nx):
            for di, dj in ((1, 0), (0, 1), (1, 1)):
                a, b = i + di, j + dj
                if a < nx and b < ny and not (apart and i < nx - apart <= a):
                    rows[j * nx + i].append(b * nx + a)
                    rows[b * nx + a].append(j * nx + i)
    rows = [rng.permutation(r) for r in rows]
    col = np.concatenate(rows).astype(np.uint32)
    rp = np.zeros(n + 1, np.uint32)
    rp[1:] = np.cumsum([len(r) for r in rows])
    at = np.repeat(np.arange(n), np.diff(rp.astype(np.int64)))
    area = rng.uniform(0.5, 1.5, n)
    area[rng.choice(n, negative, replace=False)] = -0.25
    return dict(row_ptr=rp, col=col, length=np.hypot(x[at] - x[col], y[at] - y[col]), area=area,
                erodibility=rng.uniform(0.2, 5.0, n), uplift=np.ones(n), init_elevation=rng.uniform(0, 1e-6, n),
                outlets=np.arange(0, n, nx, dtype=np.uint32), max_slope=np.full(n, 0.6) if slopes else None,
                max_iteration=40)


CASES = [(9, 7, 3, 0, False), (12, 10, 0, 3, False), (11, 12, 4, 2, True)]


@pytest.mark.parametrize("case", CASES)
def test_emulated_lasting_lakes(case):
    from cpu_emu import emu
    from test_cpu_emulation import _emu_solve

    _check(lambda ts: _emu_solve(emu.lib(), ts), [_terrain(*case, 0)])
    _check(lambda ts: _emu_solve(emu.lib(), ts), [_terrain(*case, 1), _terrain(6, 5, 0, 0, case[4], 2)])


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES + [(80, 60, 40, 0, False), (150, 100, 5, 4, False), (90, 90, 30, 3, True)])
def test_lasting_lakes(case):
    from fastlem_amd.device import DeviceBatch, DeviceTerrain

    lakes = []

    def solve(ts):
        b = DeviceBatch(ts)
        its = b.solve()
        return [b.elevations(i) for i in range(len(ts))], its

    def alone(ts):
        t = ts[0]
        d = DeviceTerrain(t["row_ptr"], t["col"], t["length"], t["area"], t["erodibility"], t["uplift"],
                          t["init_elevation"], t["outlets"], t["max_slope"], t["max_iteration"])
        it = d.solve()
        lakes.append((d.last_stats(), it))
        return [d.elevations()], [it]

    _check(alone, [_terrain(*case, 0)])
    st, it = lakes[0]
    assert st["redone"] == 0 and (st["lake_iterations"] == it or case[3] == 0)
    _check(solve, [_terrain(*case, 1), _terrain(30, 20, 0, 0, case[4], 2), _terrain(*case, 3)])
