"""The swap kernel in every shape bm_set_tuning accepts (waves per block, list
entries per lane), for listed, uniform and u-major candidates, on graphs with
narrow and wide row tables, with and without the shared contributions."""
import numpy as np
import pytest

from conftest import make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unroll", [2, 4, 8])
@pytest.mark.parametrize("waves", [1, 8])
@pytest.mark.parametrize("scale", [1, 100000])
def test_every_shape_gives_the_same_deltas(bm, orc, unroll, waves, scale):
    n = 400
    male, female, _, pi = make_pair(bm, n=n, deg=30.0, weights=bm.WEIGHTS_LOGNORMAL, seed=3)
    male, female = (bm.Graph(g.src, g.dst, g.w * scale, n) for g in (male, female))
    o = orc.Oracle(n, male, female)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        ctx.set_tuning(bm.KERNEL_SWAP, waves, 320, 8, unroll=unroll)
        assert ctx.get_tuning(bm.KERNEL_SWAP)["unroll"] == unroll
        b = ctx.batch(20000)
        for k in (7, 3000, 20000):     # the last one with the contributions summed once
            uv = orc.uniform_pairs(11, k, n)
            want = o.swap_deltas(pi, uv)
            assert np.array_equal(ctx.swap_deltas(uv), want)
            b.eval_swaps_uniform(11, k)
            assert np.array_equal(b.deltas(), want)
            b.gen_umajor(11, k)
            listed = b.pairs()
            b.eval_swaps_umajor(11, k)
            assert np.array_equal(b.deltas(), o.swap_deltas(pi, listed))
        b.close()
