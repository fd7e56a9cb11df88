"""Calls whose time must follow the work they are asked for, compared with a
second call on the same device rather than with a clock: factors of several
lie between the two sides of every comparison."""
import time

import numpy as np
import pytest
from conftest import make_pair

pytestmark = pytest.mark.gpu


def _best(prepare, call, reps=3):
    t = []
    for _ in range(reps):
        prepare()
        a = time.perf_counter()
        call()
        t.append(time.perf_counter() - a)
    return min(t)


def test_acceptance_ends_at_its_limit(bm, orc):
    """One accepted swap of 2^22 positive candidates does not walk the other
    4,095 tiles of 1,024 candidates."""
    n, k = 3000, 1 << 22
    male, female, _, pi = make_pair(bm, n=n, deg=3.0, seed=21)
    uv = orc.uniform_pairs(5, 50000, n)
    up = uv[orc.Oracle(n, male, female).swap_deltas(pi, uv) > 0]
    with bm.Context(n, male, female) as ctx:
        b = ctx.batch(k)
        b.set_pairs(np.resize(up, (k, 2)))

        def prepare():
            ctx.set_mapping(pi)
            b.eval_swaps()
            assert b.stats()["n_pos"] == k

        one = _best(prepare, lambda: b.accept_disjoint(1))
        many = _best(prepare, lambda: b.accept_disjoint(0))
        b.close()
    print(f"[costs] one {1e3 * one:.2f} ms, all {1e3 * many:.2f} ms", flush=True)
    assert one < 0.5 * many


def test_patch_of_an_accepted_batch_costs_less_than_a_build(bm):
    """Hundreds of accepted swaps of a sparse graph, a few thousand edges in
    all, are added to the table in a fraction of the time that builds it."""
    n, k = 36000, 1 << 18
    male, female, _, pi = make_pair(bm, n=n, deg=20.0, weights=bm.WEIGHTS_LOGNORMAL, seed=4)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        ctx.gain_enable(True)
        ctx.timing_enable(True)
        b = ctx.batch(k)
        patch, build = [], []
        for seed in (1, 2, 3):
            ctx.timing_reset()
            ctx.set_mapping(pi)
            b.gen_pairs(seed, k)
            b.eval_swaps()
            accepted, _ = b.accept_disjoint()
            ctx.sync()
            assert accepted > 300
            patch.append(ctx.timing(bm.KERNEL_GAIN_UPDATE)[1])
            build.append(ctx.timing(bm.KERNEL_GAIN_BUILD)[1])
        b.close()
    print(f"[costs] {accepted} swaps: patch {min(patch):.3f} ms, build {min(build):.3f} ms", flush=True)
    assert min(patch) < 0.5 * min(build)


def test_chain_shapes_are_the_ones_asked_for(bm):
    """Four waves per chain and one wave per chain can both be selected and are
    reported as what runs: with few chains and long lists the first takes about
    a third of the second's time; the chains are the same."""
    n = 4000
    male, female, _, pi = make_pair(bm, n=n, deg=200.0, weights=bm.WEIGHTS_LOGNORMAL, seed=9)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        with bm.Anneal([ctx], chains_per_instance=64, seed=3, t0=50.0, decay=0.9999, p_rot3=0.1) as ann:
            took, state = {}, {}
            for lanes, waves, unroll in ((64, 1, 4), (64, 8, 2), (256, 1, 2), (0, 1, 2)):
                ann.set_tuning(waves, 640, 16, unroll=unroll, group_lanes=lanes)
                t = ann.tuning()
                if lanes == 64:
                    assert (t["group_lanes"], t["waves_per_block"], t["unroll"]) == (64, waves, unroll)
                else:
                    assert (t["group_lanes"], t["waves_per_block"], t["unroll"]) == (256, 4, 4)

                def run():
                    ann.run(200, 1)
                    ann.state()

                took[lanes] = _best(ann.reset, run)
                state[lanes, waves] = ann.state()
            want = state[64, 1]
            for got in state.values():
                assert all(np.array_equal(got[k], want[k]) for k in want)
            best, trials = ann.autotune(steps=100)
            assert best == ann.tuning() and best["group_lanes"] == 256 and int(np.argmin(trials[:, 4])) == len(trials) - 1
    print(f"[costs] 64 lanes {1e3 * took[64]:.2f} ms, 256 lanes {1e3 * took[256]:.2f} ms", flush=True)
    assert took[256] < 0.67 * took[64]


def test_chains_of_short_lists_keep_a_wave_each(bm):
    """Unasked, chains whose steps have no entries for four waves, or that would
    take several rounds of blocks, keep one wave each."""
    n = 2000
    male, female, _, pi = make_pair(bm, n=n, deg=5.0, seed=9)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        for chains in (1, 1024):
            with bm.Anneal([ctx], chains_per_instance=chains, seed=3, t0=50.0, decay=0.9999, p_rot3=0.1) as ann:
                assert ann.tuning()["group_lanes"] == 64


def test_ranking_ties_and_its_largest_top(bm):
    """2^22 equal scores take all blocks' passes, not one block's, and 8,192
    pairs wanted cost little more than 4,096."""
    n = 2000
    male, female, _, pi = make_pair(bm, n=n, deg=20.0, seed=2)
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        with bm.Mlp(ctx, seed=1) as m:
            m.refresh_features()
            b = ctx.batch(8192)

            def took(pool, top):
                def call():
                    b.gen_learned(m, 5, pool, top)
                    ctx.sync()
                call()
                return _best(lambda: None, call, reps=5)

            half, full, plain = took(1 << 20, 4096), took(1 << 20, 8192), took(1 << 22, 4096)
            m.set_params(np.zeros(bm.Mlp.N_PARAMS, np.float32))
            ties = took(1 << 22, 4096)
            b.close()
    print(f"[costs] 4096 {1e6 * half:.0f} us, 8192 {1e6 * full:.0f} us; 2^22 {1e6 * plain:.0f} us, equal {1e6 * ties:.0f} us",
          flush=True)
    assert full < 2.5 * half
    assert ties < 4.0 * plain
