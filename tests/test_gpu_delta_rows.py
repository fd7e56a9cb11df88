"""u-major lookups from one LDS row of deltas per first vertex: complete
matchings with self-loops, u<->v edges and reversed pairs, at row lengths
around the block's and pair counts on both sides of half the square of n,
against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def graph(bm, rng, n, m, loops):
    src = rng.integers(1, n + 1, m).astype(np.int32)
    dst = rng.integers(1, n + 1, m).astype(np.int32)
    h = m // 3
    src[:h], dst[:h] = dst[h:2 * h], src[h:2 * h]      # reversed edges
    if loops:
        dst[-(m // 10):] = src[-(m // 10):]
    else:
        dst = np.where(src == dst, dst % n + 1, dst).astype(np.int32)
    return bm.Graph(src, dst, rng.integers(1, 30, m).astype(np.int32), n)


@pytest.mark.parametrize("loops", [False, True])
@pytest.mark.parametrize("n,m,k", [(2, 6, 50), (3, 9, 1), (65, 600, 9000), (1023, 30000, 530000), (2049, 30000, 2100000)])
def test_deltas_match_oracle(bm, orc, n, m, k, loops):
    rng = np.random.default_rng(n + loops)
    male, female = graph(bm, rng, n, m, loops), graph(bm, rng, n, m, loops)
    pi = np.concatenate([[0], rng.permutation(n) + 1]).astype(np.int32)
    o = orc.Oracle(n, male, female)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        ctx.gain_enable(True)
        b = ctx.batch(k)
        for seed in (1, 2):
            b.eval_swaps_umajor(seed, k)
            assert np.array_equal(b.deltas(), o.swap_deltas(pi, orc.umajor_pairs(seed, k, n)))
            ctx.apply_swap(1, 2)
            pi = ctx.get_mapping()
        b.close()
