"""Changed-first enumerations by placement rows against the oracle: packed and
wide graphs, self-loops, unmatched vertices, u <-> v edges, one changed vertex,
more than one group of them; and that lists of the same size, other
enumerations in between, shared images and moved matchings give what they
should."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 3000


def _graphs(bm, kind):
    rng = np.random.default_rng(17)

    def g(m, hubs):
        src = rng.integers(1, N + 1, m).astype(np.int32)
        dst = rng.integers(1, N + 1, m).astype(np.int32)
        src[: m // 4] = rng.integers(1, hubs, m // 4)          # a few long out-lists
        dst[m // 2: m // 2 + 500] = src[m // 2: m // 2 + 500]  # self-loops
        src[-2000:], dst[-2000:] = dst[:2000].copy(), src[:2000].copy()   # both directions
        w = rng.integers(1, 40, m).astype(np.int32)
        return bm.Graph(src, dst, w, N)

    male, female = g(500_000, 30), g(450_000, 40)
    if kind == "wide":
        female.w[::9] = rng.integers(1 << 17, 1 << 18, female.w[::9].size).astype(np.int32)
        male.w[::11] = -rng.integers(1, 30, male.w[::11].size).astype(np.int32)
    pi = np.concatenate([[0], rng.permutation(np.arange(1, N + 1))]).astype(np.int32)
    pi[rng.choice(np.arange(1, N + 1), 7, replace=False)] = 0
    if kind == "shared":
        pi[10:20] = pi[5]
    return male, female, pi


@pytest.fixture(scope="module", params=["packed", "wide", "shared"])
def setup(request, bm, orc):
    male, female, pi = _graphs(bm, request.param)
    ctx = bm.Context(N, male, female)
    ctx.set_mapping(pi)
    yield ctx, orc.Oracle(N, male, female), pi
    ctx.close()


def _changed(pi, c):
    rng = np.random.default_rng(c)
    ch = rng.choice(np.arange(1, N + 1), c, replace=False)
    ch[0] = 3                                   # a hub
    if c > 3:
        ch[1] = int(np.flatnonzero(pi[1:] == 0)[0]) + 1   # an unmatched vertex
    return np.unique(ch)[::-1].astype(np.int32)


@pytest.mark.parametrize("c", [1, 4, 40, 140])
def test_pairs(setup, c):
    ctx, o, pi = setup
    ctx.set_mapping(pi)
    d, uv = ctx.swap_deltas_changed(_changed(pi, c))
    assert np.array_equal(d, o.swap_deltas(pi, uv))


@pytest.mark.parametrize("c", [1, 2, 5])
def test_triples(setup, c):
    ctx, o, pi = setup
    ctx.set_mapping(pi)
    best, q = ctx.rot3_deltas_changed(_changed(pi, c))
    want, perm = o.rot3_many(pi, q[:, :3])
    assert np.array_equal(best, want) and np.array_equal(q[:, 3], perm)


def test_list_after_enumeration_and_moves(setup, orc):
    ctx, o, pi = setup
    ctx.set_mapping(pi)
    ch = _changed(pi, 40)
    b = ctx.batch(40 * N)
    other = ctx.batch(40 * N)
    b.gen_changed_pairs(ch)
    other.gen_changed_pairs(ch[:7])             # another enumeration of the same context in between
    b.eval_swaps()
    uv = b.pairs()
    assert np.array_equal(b.deltas(), o.swap_deltas(pi, uv))
    ctx.apply_swap(int(ch[0]), int(ch[1]))      # the same list under the moved matching
    moved = ctx.get_mapping()
    b.eval_swaps()
    assert np.array_equal(b.deltas(), o.swap_deltas(moved, uv))
    lst = orc.uniform_pairs(3, len(uv), N)      # a list of the same length is not an enumeration
    b.set_pairs(lst)
    b.eval_swaps()
    assert np.array_equal(b.deltas(), o.swap_deltas(moved, lst))
    b.close()
    other.close()
