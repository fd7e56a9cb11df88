"""More vertices than one launch of a block each can cover (2^24 rows of 256
threads): every row table is filled."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_row_tables_of_more_than_two_to_the_24_rows(bm):
    n, m = (1 << 24) + 10, 4000
    rng = np.random.default_rng(1)
    src = rng.integers(1, n + 1, m).astype(np.int32)
    dst = rng.integers(1, n + 1, m).astype(np.int32)
    src[:10], dst[:10] = n, np.arange(1, 11)
    src[10:20], dst[10:20] = np.arange(1, 11), n - 1
    w = rng.integers(1, 9, m).astype(np.int32)
    weight = {(int(a), int(b)): int(x) for a, b, x in zip(src, dst, w)}     # the last line counts
    g = bm.Graph(src, dst, w, n)
    uv = np.array([[n, 5], [1, 2], [int(src[100]), int(dst[200])], [n, n - 1], [3, int(dst[300])]], np.int32)

    def score(swap):
        to = {swap[0]: swap[1], swap[1]: swap[0]} if swap is not None else {}
        return sum(min(x, weight.get((to.get(a, a), to.get(b, b)), 0)) for (a, b), x in weight.items())

    now = score(None)
    with bm.Context(n, g, g) as ctx:
        ctx.set_mapping(np.arange(n + 1, dtype=np.int32))
        assert ctx.score() == now
        assert ctx.swap_deltas(uv).tolist() == [score([int(a), int(b)]) - now for a, b in uv]
        with bm.Anneal([ctx], chains_per_instance=2, seed=1) as ann:
            ann.run(20, 1)
            assert ann.verify() == 0
