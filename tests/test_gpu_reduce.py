"""Batch statistics and the rank-th pick over sizes at the edges of the
chunks: one chunk (no partial results), a ragged last chunk, and the sizes at
which the chunk doubles."""
import numpy as np
import pytest

from conftest import make_pair

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(bm):
    male, female, _, pi0 = make_pair(bm, n=300, deg=12.0, seed=17)
    c = bm.Context(300, male, female)
    c.set_mapping(pi0)
    yield c
    c.close()


@pytest.mark.parametrize("k", [1, 2, 63, 255, 4095, 4096, 4097, 8192 + 17, (1 << 20) + 4095, 1 << 25, (1 << 25) + 1,
                               (1 << 26) - 3])
def test_stats_and_pick(ctx, k):
    b = ctx.batch(k)
    try:
        b.gen_pairs(1000 + k, k)
        b.eval_swaps()
        d = b.deltas()
        st = b.stats()
        assert st["count"] == k
        assert st["sum"] == int(d.sum())
        assert st["max"] == int(d.max())
        assert st["argmax"] == int(d.argmax())
        assert st["n_pos"] == int((d > 0).sum())
        assert st["n_zero"] == int((d == 0).sum())
        for kind, hits in ((1, np.flatnonzero(d > 0)), (0, np.flatnonzero(d == 0))):
            for rank in sorted({0, len(hits) // 2, len(hits) - 1} - {-1}):
                if rank < len(hits):
                    assert b.pick(kind, rank) == hits[rank], (kind, rank)
            assert b.pick(kind, len(hits)) == -1
    finally:
        b.close()
