"""Table patches by row owner: one move list past a block's slots, female rows
past one unit, and graphs smaller and larger than the grid."""
import numpy as np
import pytest

from conftest import make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,deg,k", [(5, 2.0, 10), (700, 300.0, 20000), (2500, 10.0, 40000)])
def test_accepted_batch_patches_every_row(bm, n, deg, k):
    male, female, _, pi0 = make_pair(bm, n=n, deg=deg, seed=n)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi0)
        ctx.gain_enable(True)
        b = ctx.batch(k)
        for seed in (1, 2):
            b.gen_pairs(seed, k)
            b.eval_swaps()
            b.accept_disjoint()
        ctx.apply_swap(1, n)
        ctx.apply_perm3(1, 2, n, 3)
        b.close()
        patched = np.array([ctx.gain_row(u) for u in range(1, n + 1)])
        pi = ctx.get_mapping()
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        ctx.gain_enable(True)
        built = np.array([ctx.gain_row(u) for u in range(1, n + 1)])
    assert not np.array_equal(pi, pi0)
    assert np.array_equal(patched, built)
