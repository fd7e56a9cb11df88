"""The learned ranking where thousands of scores are equal: every digit the
select can need, from the score's last bits to the fine place in pools past
2^25 pairs, against a stable sort."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def net(bm):
    n = 700
    male, female, _, pi = bm.synth_pair(n, 15.0, bm.WEIGHTS_GEOMETRIC, 0.3, seed=9)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        with bm.Mlp(ctx, seed=1) as m:
            m.refresh_features()
            yield ctx, m


def _params(bm, slope, bias):
    p = np.zeros(bm.Mlp.N_PARAMS, np.float32)
    w1, b1, w2, b2, w3, b3 = bm.Mlp.unpack(p)
    w1[0, 0], w2[0, 0], w3[0], b3[0] = 1.0, 1.0, slope, bias
    return p


@pytest.mark.parametrize("pool,top", [(8193, 8192), (16385, 1), (1 << 20, 4096), (1 << 25, 8192), ((1 << 25) + 5, 8192),
                                      ((1 << 26) + 3, 17)])
def test_equal_scores_keep_the_pool_order(bm, orc, net, pool, top):
    ctx, m = net
    m.set_params(_params(bm, 0.0, 0.25))
    b = ctx.batch(top)
    b.gen_learned(m, 31, pool, top)
    assert np.array_equal(b.pairs(), orc.uniform_pairs(31, top, ctx.n))
    b.close()


# a slope of 2^-19 on a score of 1/4 separates values only in its last 8 bits
@pytest.mark.parametrize("slope", [1.0, 2.0 ** -19])
@pytest.mark.parametrize("pool,top", [(300001, 8192), (300001, 100), (1 << 20, 5000), (20000, 8192)])
def test_few_distinct_scores(bm, orc, net, pool, top, slope):
    ctx, m = net
    m.set_params(_params(bm, slope, 0.25))
    stream = orc.uniform_pairs(77, pool, ctx.n)
    score = m.score_pairs(stream)
    want = stream[np.argsort(-score.astype(np.float64), kind="stable")[:top]]
    b = ctx.batch(top)
    b.gen_learned(m, 77, pool, top)
    assert np.array_equal(b.pairs(), want)
    b.gen_learned_noalloc(m, 77, pool, top)
    assert np.array_equal(b.pairs(), want)
    b.close()
