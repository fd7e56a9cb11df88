"""Disjoint acceptance at the edges of its two orderings (small batches ranked
by counting, large ones sorted) and of its rounds of 16: batch sizes around the
limits, ties, deltas beyond 32 bits, many rejected candidates in a row, a
max_accept inside a round; always the oracle's sequential greedy."""
import numpy as np
import pytest
from conftest import make_pair, quirky_pair

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sparse(bm, orc):
    n = 3000
    male, female, _, pi = make_pair(bm, n=n, deg=3.0, seed=21)
    return n, male, female, pi, orc.Oracle(n, male, female)


def _deltas(kind, rng, k):
    if kind == "ties":
        return rng.integers(-1, 3, k).astype(np.int64)
    if kind == "wide":
        return rng.integers(-(1 << 50), 1 << 50, k).astype(np.int64)
    return np.where(rng.random(k) < 0.02, rng.integers(1, 1000, k), 0).astype(np.int64)


@pytest.mark.parametrize("kind", ["ties", "wide", "few"])
@pytest.mark.parametrize("k", [1, 15, 16, 17, 1025, 4096, 8191, 8192, 8193, 20000])
def test_accept_matches_sequential_greedy(bm, sparse, kind, k):
    n, male, female, pi, o = sparse
    rng = np.random.default_rng(k)
    uv = np.stack([rng.integers(1, n + 1, k), rng.integers(1, n + 1, k)], axis=1).astype(np.int32)
    uv[: k // 3, 0] = rng.integers(1, 20, k // 3)      # a few vertices in many candidates: long runs of rejections
    d = _deltas(kind, rng, k)
    want_pi, want_acc, want_gain = o.accept_disjoint(pi, uv, d)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        acc, gain = ctx.accept_disjoint(uv, d)
        assert np.array_equal(acc, want_acc) and gain == want_gain
        assert np.array_equal(ctx.get_mapping(), want_pi)
        # the inverse matching moved along: deltas after the acceptance
        q = uv[: min(k, 200)]
        assert np.array_equal(ctx.swap_deltas(q), o.swap_deltas(want_pi, q))


@pytest.mark.parametrize("limit", [1, 3, 16, 17, 40])
def test_max_accept_cuts_the_same_sequence(bm, orc, sparse, limit):
    n, male, female, pi, o = sparse
    k = 4000
    uv = orc.uniform_pairs(5, k, n)
    d = o.swap_deltas(pi, uv)
    want, acc, gain = o.accept_disjoint(pi, uv, d, limit)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        b = ctx.batch(k)
        b.set_pairs(uv)
        b.eval_swaps()
        assert b.accept_disjoint(limit) == (len(acc), gain)
        assert np.array_equal(ctx.get_mapping(), want)
        b.close()


def test_accept_with_unmatched_and_self_loops(bm, orc):
    male, female, pi = quirky_pair(bm)
    n = 60
    o = orc.Oracle(n, male, female)
    uv = orc.uniform_pairs(3, 900, n)
    d = o.swap_deltas(pi, uv)
    want_pi, want_acc, want_gain = o.accept_disjoint(pi, uv, d)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        acc, gain = ctx.accept_disjoint(uv, d)
        assert np.array_equal(acc, want_acc) and gain == want_gain and np.array_equal(ctx.get_mapping(), want_pi)
        assert np.array_equal(ctx.swap_deltas(uv), o.swap_deltas(want_pi, uv))
