"""The learned ranking's select: a pool's leading pairs equal a stable
descending sort of the pool's scores, whatever ties there are (the two digits
that settle most pools, the further digits when thousands of scores share
them, the largest `top`, and pools smaller than a wave)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _network(bm, kind):
    p = np.zeros(bm.Mlp.N_PARAMS, np.float32)
    w1, b1, w2, b2, w3, b3 = bm.Mlp.unpack(p)
    rng = np.random.default_rng(5)
    if kind == "random":
        w1[...] = rng.normal(size=w1.shape) * 0.3
        w2[...] = rng.normal(size=w2.shape) * 0.1
        w3[...] = rng.normal(size=w3.shape) * 0.1
    elif kind == "degree":      # the score is u's log out-degree: long runs of equal scores
        w1[0, 0], w2[0, 0], w3[0] = 1.0, 1.0, 1.0
    b3[0] = {"equal": 0.0, "negative": -2.5}.get(kind, 0.125)
    return p


@pytest.fixture(scope="module")
def net(bm):
    n = 700
    male, female, _, pi = bm.synth_pair(n, 15.0, bm.WEIGHTS_GEOMETRIC, 0.3, seed=9)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        with bm.Mlp(ctx, seed=1) as m:
            m.refresh_features()
            yield ctx, m


@pytest.mark.parametrize("kind", ["random", "degree", "equal", "negative"])
@pytest.mark.parametrize("pool,top", [(1, 1), (63, 63), (5000, 17), (40001, 4096), (40001, 8191), (70000, 8192),
                                      (8192, 8192)])
def test_select_is_a_stable_sort(bm, orc, net, kind, pool, top):
    ctx, m = net
    m.set_params(_network(bm, kind))
    stream = orc.uniform_pairs(77, pool, ctx.n)
    score = m.score_pairs(stream)
    want = stream[np.argsort(-score.astype(np.float64), kind="stable")[:top]]
    b = ctx.batch(top)
    b.gen_learned(m, 77, pool, top)
    assert np.array_equal(b.pairs(), want)
    b.gen_learned_noalloc(m, 77, pool, top)
    assert np.array_equal(b.pairs(), want)
    b.close()
