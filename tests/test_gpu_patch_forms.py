"""Table patches by work items and by rows, with the transposed copy patched
alongside: after moves of ordinary vertices, hubs and a whole accepted batch
the table and the best partners (which read both copies) are those of a table
built from the matching."""
import numpy as np
import pytest

from conftest import make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,deg,k", [(900, 12.0, 3000), (900, 40.0, 200), (3000, 8.0, 9000)])
def test_both_forms_keep_both_copies(bm, n, deg, k):
    male, female, _, pi0 = make_pair(bm, n=n, deg=deg, weights=bm.WEIGHTS_LOGNORMAL, seed=n)
    d = np.bincount(male.src, minlength=n + 1) + np.bincount(male.dst, minlength=n + 1)
    order = np.argsort(d[1:], kind="stable") + 1      # light vertices first, hubs last
    light, mid, hubs = order[:6], order[n // 2:n // 2 + 6], order[-6:]

    def state(ctx):
        rows = np.array([ctx.gain_row(u) for u in range(1, n + 1)])
        return rows, ctx.best_partners(1, n)

    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi0)
        ctx.gain_enable(True)
        seen = []
        for vs in (light, mid, hubs, (light[0], hubs[0], mid[0], hubs[1], mid[1], light[1])):
            vs = [int(v) for v in vs]
            ctx.best_partners(1, n)                   # the transposed copy is current before the moves
            ctx.apply_swap(vs[0], vs[1])
            ctx.apply_perm3(vs[2], vs[3], vs[4], 3)
            ctx.apply_swap(vs[5], vs[0])
            seen.append((ctx.get_mapping(), state(ctx)))
        b = ctx.batch(k)
        b.gen_pairs(3, k)
        b.eval_swaps()
        assert b.accept_disjoint()[0] > 0
        b.close()
        seen.append((ctx.get_mapping(), state(ctx)))
    with bm.Context(n, male, female) as ctx:
        ctx.gain_enable(True)
        for pi, (rows, partners) in seen:
            ctx.set_mapping(pi)
            want_rows, want_partners = state(ctx)
            assert np.array_equal(rows, want_rows)
            for a, b in zip(partners, want_partners):
                assert np.array_equal(a, b)
