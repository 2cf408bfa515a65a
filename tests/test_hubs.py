"""Sites with more neighbours than are loaded or listed together: hubs whose rows
end around 8, 64 and 128 entries and far past them, some of their children heads of
chains, as outlets, inside a long chain and in its short ones.  Bit for bit against
the oracle, on the GPU and in the CPU emulation; and a hub's row of 20 000 entries
costs the permutation and the drainage-area sweep about what it costs the kernel
that looks for its children."""
import ctypes

import numpy as np
import pytest

from test_sweeps import _check


def _hubs(kids, spine, slopes, seed):
    """A path of `spine` sites from the outlet on; every third one (the outlet, too)
    has `kids` further children, every fourth of them a child of its own; the rows in
    random order."""
    rng = np.random.default_rng([kids, spine, seed])
    parent = list(range(-1, spine - 1))
    for s in range(0, spine, 3):
        for k in range(kids):
            parent.append(s)
            if k % 4 == 3:
                parent.append(len(parent) - 1)
    parent, n = np.array(parent), len(parent)
    h = np.zeros(n)
    length = rng.uniform(0.5, 1.5, n)
    for v in range(1, n):
        h[v] = h[parent[v]] + rng.uniform(0.1, 1.0)
    a = np.r_[np.arange(1, n), parent[1:]]
    b = np.r_[parent[1:], np.arange(1, n)]
    order = np.lexsort((rng.random(len(a)), a))
    return dict(row_ptr=np.r_[0, np.cumsum(np.bincount(a, minlength=n))].astype(np.uint32), col=b[order].astype(np.uint32),
                length=np.r_[length[1:], length[1:]][order], area=rng.uniform(0.1, 3.0, n),
                erodibility=rng.uniform(0.2, 5.0, n), uplift=rng.uniform(0.1, 2.0, n), init_elevation=h,
                outlets=np.array([0], np.uint32), max_slope=np.full(n, 0.6) if slopes else None, max_iteration=4)


KIDS = (6, 7, 8, 9, 10, 61, 62, 63, 64, 65, 126, 127, 129, 300)


@pytest.mark.parametrize("slopes", [False, True])
def test_emulated_hubs(slopes):
    from cpu_emu import emu
    from test_cpu_emulation import _emu_solve

    for kids in KIDS:
        _check(lambda ts: _emu_solve(emu.lib(), ts), [_hubs(kids, 4, slopes, 0)])
    _check(lambda ts: _emu_solve(emu.lib(), ts), [_hubs(9, 140, slopes, 1), _hubs(66, 40, slopes, 2)])


@pytest.mark.gpu
@pytest.mark.parametrize("slopes", [False, True])
def test_hubs(slopes):
    from fastlem_amd.device import DeviceBatch

    def solve(ts):
        b = DeviceBatch(ts)
        its = b.solve()
        return [b.elevations(i) for i in range(len(ts))], its

    _check(solve, [_hubs(k, s, slopes, 3) for k in KIDS for s in (1, 4, 20)])
    for kids, spine in ((9, 140), (66, 300), (5000, 4), (20, 1000)):
        _check(solve, [_hubs(kids, spine, slopes, 4)])


@pytest.mark.gpu
def test_time_of_a_hub():
    from fastlem_amd import _native
    from fastlem_amd.device import DeviceTerrain
    from fastlem_amd.generator import context

    L, ctx, k = _native.lib(), context(), 20_000
    n, rng = k + 1, np.random.default_rng(0)
    length, one = rng.uniform(0.5, 1.5, k), np.ones(k + 1)
    d = DeviceTerrain(np.r_[0, k + np.arange(k + 1)].astype(np.uint32), np.r_[np.arange(1, n), np.zeros(k)].astype(np.uint32),
                      np.r_[length, length], one, one, one, np.r_[0.0, rng.uniform(0.0, 1.0, k)], np.array([0], np.uint32))
    d.solve()
    _native.check(L.fl_ctx_set_profiling(ctx, 1))
    try:
        _native.check(L.fl_ctx_reset_profile(ctx))
        for _ in range(3):
            d.solve()

        def ms(*names):
            total = 0.0
            for name in names:
                c, t, u = ctypes.c_uint64(), ctypes.c_double(), ctypes.c_uint64()
                _native.check(L.fl_ctx_kernel_time(ctx, name.encode(), ctypes.byref(c), ctypes.byref(t), ctypes.byref(u)))
                total += t.value
            return total

        children, perm, area = ms("k_children"), ms("k_chain_perm"), ms("k_da_fold", "k_da_tail")
    finally:
        L.fl_ctx_set_profiling(ctx, 0)
        d.close()
    print(f"k_children {children:.2f} ms, k_chain_perm {perm:.2f}, drainage area {area:.2f}")
    assert perm < 3 * children and area < 3 * children, (children, perm, area)
