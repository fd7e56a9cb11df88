"""The list-intersection swap kernel over the forms it takes: packed and wide
row tables, matchings with shared and missing images (no inverse: the male
side only), self-loops and u <-> v edges, batches below and above the limits
of its two launch shapes and of the shared current contributions, and the
matching moved by every kind of move (its inverse moves along)."""
import numpy as np
import pytest
from conftest import make_pair, quirky_pair

pytestmark = pytest.mark.gpu


def _variant(bm, kind):
    """(n, male, female, pi) whose weights or matching force one form."""
    if kind == "quirky":
        male, female, pi = quirky_pair(bm, n=60, m=700)
        return 60, male, female, pi
    n = 400
    male, female, _, pi = make_pair(bm, n=n, deg=25.0, seed=31)
    rng = np.random.default_rng(2)
    if kind == "negative_male":
        male.w[::7] = -rng.integers(1, 50, male.w[::7].size).astype(np.int32)
    elif kind == "wide_weights":
        female.w[::5] = rng.integers(1 << 20, 1 << 30, female.w[::5].size).astype(np.int32)
        male.w[::3] = rng.integers(1 << 20, 1 << 30, male.w[::3].size).astype(np.int32)
    elif kind == "shared_images":
        pi[rng.choice(np.arange(1, n + 1), 40, replace=False)] = pi[7]
        pi[rng.choice(np.arange(1, n + 1), 10, replace=False)] = 0
    elif kind == "empty_rows":
        keep = (male.src % 3 != 0) & (male.dst % 5 != 0)
        male = bm.Graph(male.src[keep], male.dst[keep], male.w[keep], n)
    return n, male, female, pi


@pytest.mark.parametrize("kind", ["plain", "quirky", "negative_male", "wide_weights", "shared_images", "empty_rows"])
@pytest.mark.parametrize("k", [1, 3, 300, 40000])
def test_swap_deltas_every_form(bm, orc, kind, k):
    n, male, female, pi = _variant(bm, kind)
    o = orc.Oracle(n, male, female)
    uv = orc.uniform_pairs(11, k, n)
    uv[k // 2] = (5, 5)
    want = o.swap_deltas(pi, uv)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        assert ctx.score() == o.score(pi)
        assert np.array_equal(ctx.swap_deltas(uv), want)
        b = ctx.batch(k)
        b.eval_swaps_uniform(11, k)
        assert np.array_equal(b.deltas(), o.swap_deltas(pi, orc.uniform_pairs(11, k, n)))
        b.eval_swaps_umajor(12, k)
        assert np.array_equal(b.deltas(), o.swap_deltas(pi, orc.umajor_pairs(12, k, n)))
        b.close()


@pytest.mark.parametrize("kind", ["plain", "quirky", "shared_images"])
def test_moves_keep_the_inverse(bm, orc, kind):
    n, male, female, pi = _variant(bm, kind)
    o = orc.Oracle(n, male, female)
    uv = orc.uniform_pairs(13, 500, n)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        for u, v in ((1, 2), (3, 9), (9, 2), (4, 4), (17, 5)):
            ctx.apply_swap(u, v)
        for p in range(6):
            ctx.apply_perm3(10 + p, 20 + p, 30 + p, p)
        assert np.array_equal(ctx.swap_deltas(uv), o.swap_deltas(ctx.get_mapping(), uv))


@pytest.mark.parametrize("n", [2, 3, 5])
def test_smallest_graphs(bm, orc, n):
    src = np.array([1, 2, 1], np.int32)
    dst = np.array([2, 1, 1], np.int32)
    male = bm.Graph(src, dst, np.array([3, 5, 2], np.int32), n)
    female = bm.Graph(src, dst, np.array([4, 1, 7], np.int32), n)
    pi = np.arange(n + 1, dtype=np.int32)
    uv = np.array([(1, 2), (2, 1), (1, 1), (1, n), (n, 2)], np.int32)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        assert np.array_equal(ctx.swap_deltas(uv), orc.Oracle(n, male, female).swap_deltas(pi, uv))


@pytest.mark.parametrize("kind", ["plain", "quirky", "negative_male", "wide_weights", "shared_images", "empty_rows"])
@pytest.mark.parametrize("k", [1, 200, 33000])
def test_triples_every_form(bm, orc, kind, k):
    n, male, female, pi = _variant(bm, kind)
    o = orc.Oracle(n, male, female)
    rng = np.random.default_rng(4)
    abc = np.stack([rng.permutation(np.arange(1, n + 1))[:3] for _ in range(k)]).astype(np.int32)
    want_b, want_p = o.rot3_many(pi, abc)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        best, perm = ctx.rot3_deltas(abc)
        assert np.array_equal(best, want_b) and np.array_equal(perm.astype(np.int32), want_p)


@pytest.mark.parametrize("per_instance", [3, 1400])
def test_chains_over_mixed_instances(bm, orc, per_instance):
    """Instances with packed and with wide row tables, with and without an
    inverse matching, in one launch: four waves per chain and (many chains)
    one; every chain's recount agrees and one of each instance replays."""
    parts = [_variant(bm, k) for k in ("plain", "wide_weights", "shared_images")]
    ctxs = []
    for n, male, female, pi in parts:
        c = bm.Context(n, male, female)
        c.set_mapping(pi)
        ctxs.append(c)
    with bm.Anneal(ctxs, chains_per_instance=per_instance, seed=6, t0=20.0, decay=0.999, p_rot3=0.3) as ann:
        for _ in range(2):          # the second time after a reset
            ann.run(40, 2)
            assert ann.verify() == 0
            st = ann.state()
            beta0, lam, p3 = ann.schedule()
            for i, (n, male, female, pi) in enumerate(parts):
                c = i * per_instance + per_instance // 2
                o = orc.Oracle(n, male, female)
                got, _, rs = orc.anneal_chain(o, pi, o.score(pi), orc.chain_seed(6, c), 0, 80, beta0, lam, p3)
                assert rs[0] == st["score"][c] and rs[1] == st["best"][c]
                assert np.array_equal(got, ann.mapping(c))
            ann.reset()
    for c in ctxs:
        c.close()
