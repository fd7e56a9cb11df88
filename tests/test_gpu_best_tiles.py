"""Best swap by table tiles (complete matchings) against the oracle, at sizes
around the 64-wide tiles, with self-loops and both edge directions, from hardly
any to all pairs adjacent, and along a climb that patches the table."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(bm, n, density, seed):
    rng = np.random.default_rng(seed)

    def g():
        a = rng.random((n + 1, n + 1)) < density
        a[0, :] = a[:, 0] = False
        a[1, min(2, n)] = True
        src, dst = np.nonzero(a)
        return bm.Graph(src.astype(np.int32), dst.astype(np.int32), rng.integers(1, 30, src.size).astype(np.int32), n)

    pi = np.concatenate([[0], rng.permutation(np.arange(1, n + 1))]).astype(np.int32)
    return g(), g(), pi


@pytest.mark.parametrize("density", [0.0, 0.1, 0.6, 1.0])
@pytest.mark.parametrize("n", [2, 31, 32, 63, 64, 65, 127, 128, 200])
def test_best_swap_by_tiles(bm, orc, n, density):
    male, female, pi = _pair(bm, n, density, 100 * n + int(10 * density))
    o = orc.Oracle(n, male, female)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        ctx.gain_enable(True)
        assert ctx.best_swap() == o.best_swap(pi)
        trace, res = ctx.best_swap_climb(6, verify_every=1)
        want_pi, want = o.best_swap_climb(pi, 6)
        assert np.array_equal(trace, want) and res["verify_failures"] == 0
        assert np.array_equal(ctx.get_mapping(), want_pi)
        pi2 = want_pi.copy()
        pi2[1 + n // 2] = 0             # an unmatched vertex: the other search, same answer
        ctx.set_mapping(pi2)
        assert ctx.best_swap() == o.best_swap(pi2)
        ctx.set_mapping(pi)
        assert ctx.best_swap() == o.best_swap(pi)
