"""bench.py's byte model: what a kernel must move for leaves is what it does for
them."""
import pytest


@pytest.mark.parametrize("clamp", [False, True])
def test_leaves(clamp):
    import bench

    def bpu(name, active, chain):
        return bench.kernel_bytes_per_unit(name, 1000, 6000, clamp, active, chain)

    # leaves take no part in pointer jumping, and leave the permutation after a few words
    assert bpu("k_chain_jump", 0.5, 0.0) == bpu("k_chain_jump", 0.0, 0.0) == 1
    assert bpu("k_chain_jump", 0.5, 0.2) == 1 + 0.2 * 32
    assert bpu("k_chain_perm", 0.3, 0.0) == 1 + 0.3 * 40
    assert bpu("k_chain_perm", 0.3, 0.1) < 0.6 * bpu("k_chain_perm", 0.3, 0.3)
    # each leaf is a word of its receiver's list, read and given back, and a step of the scatter's
    assert bpu("k_da_fold", 0.3, 0.1) - bpu("k_da_fold", 0.1, 0.1) == pytest.approx(32)
    assert bpu("k_tau_scatter", 0.3, 0.1) > bpu("k_tau_scatter", 0.3, 0.3)
    # (a chain fraction above the recomputed one is the recomputed one)
    assert bpu("k_chain_perm", 0.3, 1.0) == bpu("k_chain_perm", 0.3, 0.3)
