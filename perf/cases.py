"""The work that users of this framework have it do, as cases that can be timed.

Each case goes through the ctypes binding (brain-match_amd/brainmatch.py), the
way the tools, the drivers and the benchmark call the library.  Sizes follow
the benchmark configurations (bench.py, tests/test_gpu_configs.py): the small
pair (n = 2,000, ~40k edges, geometric weights), the full-size pair
(n = 18,524, ~4M edges, lognormal weights), uneven batched annealing
instances, the learned proposal on the full-size pair, and a wide pair whose
table rows need more than one LDS window.  `draw` spreads over the same ranges.
"""
import math
import os
import sys

import numpy as np

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "brain-match_amd"))

import brainmatch as bm  # noqa: E402

FULL_N, FULL_DEG = 18524, 4e6 / 18524


def listed():
    return [
        # one short list of pairs from the host, deltas back: a caller that
        # replaces a handful of calculate_swap_delta calls; all latency
        {"name": "list_small", "kind": "list", "n": 2000, "deg": 20.0, "geometric": True, "k": 64},
        # the enumeration of a few changed vertices with every delta and pair
        # read back, as the reference's host scan has them
        {"name": "changed_full", "kind": "changed", "n": FULL_N, "deg": FULL_DEG, "geometric": False, "c": 13},
        # graph-re-alignment-gpu-swap: one score-weighted perturbation's whole
        # enumeration (about 3.7M pairs), then the walk's steps (37k pairs each)
        {"name": "tool_swap", "kind": "search", "mode": 0, "n": FULL_N, "deg": FULL_DEG, "geometric": False,
         "iters": 24},
        # graph-re-alignment-gpu-3-swap: a uniform perturbation's triples, then
        # the walk's steps (three changed vertices each)
        {"name": "tool_rot3", "kind": "search", "mode": 2, "n": FULL_N, "deg": FULL_DEG, "geometric": False,
         "iters": 8},
        # the small configuration's greedy disjoint-swap hill climbing: short rounds
        {"name": "climb_small", "kind": "climb", "n": 2000, "deg": 20.0, "geometric": True, "rounds": 50,
         "batch": 4096},
        # climb rounds with the learned proposal: 2^20 uniform pairs ranked by
        # the network, the top 4,096 evaluated exactly
        {"name": "climb_learned", "kind": "learned", "n": FULL_N, "deg": FULL_DEG, "geometric": False, "rounds": 8,
         "pool": 1 << 20, "top": 4096},
        # the proposal network: forward scores, a gradient, training steps on
        # batches labelled by the exact kernel
        {"name": "mlp_train", "kind": "mlp", "n": FULL_N, "deg": FULL_DEG, "geometric": False, "k": 1 << 16,
         "steps": 8},
        # the benchmark's step: a new matching (table build), 2^28 uniform
        # pairs, the statistics; the deltas stay on the device, as in the
        # drivers, which read back the statistics and the candidate they pick
        {"name": "table_pairs", "kind": "table", "n": FULL_N, "deg": FULL_DEG, "geometric": False, "k": 1 << 28},
        # the same step on 2^26 uniform triples
        {"name": "table_triples", "kind": "table3", "n": FULL_N, "deg": FULL_DEG, "geometric": False, "k": 1 << 26},
        # a pair too wide for one LDS window: table build in column windows,
        # bitmap-only lookups, every delta read back
        {"name": "table_wide", "kind": "table", "n": 50000, "deg": 40.0, "geometric": False, "k": 1 << 20},
        # the score-lookup driver's loop: steepest ascent over all pairs
        {"name": "best_swap", "kind": "best", "n": FULL_N, "deg": FULL_DEG, "geometric": False, "iters": 32},
        # batched annealing: uneven instances, many chains, one launch
        {"name": "anneal", "kind": "anneal", "sizes": "1013,1999,3001,5003", "deg": 200.0, "geometric": False,
         "chains": 256, "steps": 200, "launches": 2, "p_rot3": 0.1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["list", "changed", "changed3", "search", "climb", "learned", "mlp", "table", "table3", "best", "anneal"])
    geometric = rng.random() < 0.25
    n = _log(rng, 2000, FULL_N)
    deg = round(math.exp(rng.uniform(math.log(20.0), math.log(FULL_DEG))), 2)
    c = {"kind": kind, "n": n, "deg": deg, "geometric": geometric}
    if kind == "list":
        c["k"] = _log(rng, 16, 1 << 16)
    elif kind == "changed":
        c["c"] = _log(rng, 1, 40)
    elif kind == "changed3":
        c["c"] = rng.randint(1, 5)
    elif kind == "search":
        c["mode"] = rng.choice([0, 1, 2])
        c["iters"] = rng.randint(4, 8 if c["mode"] == 2 else 24)
    elif kind == "climb":
        c["rounds"], c["batch"] = rng.randint(4, 32), _log(rng, 512, 1 << 14)
    elif kind == "learned":
        c["rounds"], c["pool"] = rng.randint(2, 8), _log(rng, 1 << 16, 1 << 20)
        c["top"] = rng.randint(512, 4096)
    elif kind == "mlp":
        c["k"], c["steps"] = 256 * rng.randint(16, 256), rng.randint(2, 8)
    elif kind == "table":
        if rng.random() < 0.3:      # beyond the single LDS window
            c["n"], c["deg"] = rng.randint(41000, 60000), round(rng.uniform(20.0, 40.0), 2)
        c["k"] = _log(rng, 1 << 16, 1 << 28)
    elif kind == "table3":
        c["k"] = _log(rng, 1 << 16, 1 << 26)
    elif kind == "best":
        c["iters"] = rng.randint(4, 32)
    elif kind == "anneal":
        c = {"kind": kind, "sizes": ",".join(str(_log(rng, 1000, 5000)) for _ in range(rng.randint(1, 4))),
             "deg": deg, "geometric": geometric, "chains": rng.randint(16, 256), "steps": rng.randint(50, 200),
             "launches": rng.randint(1, 2), "p_rot3": rng.choice([0.0, 0.1, 0.25])}
    return c


#: Above this many candidates a program reads back statistics and picks, not every delta.
WHOLE = 1 << 21


def _pair(case, n, seed):
    weights = bm.WEIGHTS_GEOMETRIC if case["geometric"] else bm.WEIGHTS_LOGNORMAL
    male, female, _, pi = bm.synth_pair(n, case["deg"], weights, 0.3, seed=seed)
    return male, female, pi


def _uniform_pairs(rng, n, k):
    u = rng.integers(1, n + 1, k)
    v = rng.integers(1, n, k)
    return np.stack([u, v + (v >= u)], axis=1).astype(np.int32)


def _host_inputs(case, seed):
    """What both prepare and exact start from."""
    rng = np.random.default_rng(seed)
    male, female, pi = _pair(case, case["n"], seed + 1)
    s = {"male": male, "female": female, "pi": pi}
    if case["kind"] in ("changed", "changed3"):
        s["changed"] = rng.choice(np.arange(1, case["n"] + 1), case["c"], replace=False).astype(np.int32)
    if case["kind"] in ("list", "mlp"):
        s["uv"] = _uniform_pairs(rng, case["n"], case["k"])
    if case["kind"] == "mlp":
        # labels as training sees them: sign(d) log1p|d| of heavy-tailed deltas
        s["target"] = (rng.normal(size=case["k"]) * 3.0).astype(np.float32)
        p = []
        for a, b in ((16, 128), (128, 128), (128, 1)):
            p += [(rng.normal(size=(a, b)) * math.sqrt(2.0 / a)).astype(np.float32).ravel(),
                  (rng.normal(size=b) * 0.01).astype(np.float32)]
        s["params"] = np.concatenate(p)
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "anneal":
        ctxs = []
        for i, n in enumerate(int(x) for x in case["sizes"].split(",")):
            male, female, pi = _pair(case, n, seed + 1 + 1000 * i)
            ctx = bm.Context(n, male, female)
            ctx.set_mapping(pi)
            ctxs.append(ctx)
        a = bm.Anneal(ctxs, chains_per_instance=case["chains"], seed=seed + 5, t0=50.0, decay=0.9999,
                      p_rot3=case["p_rot3"], traj_cap=case["launches"])
        a.set_tuning(1, 2560, 16, unroll=2)    # the shape the autotuner keeps for such instances
        return {"case": case, "anneal": a}
    s = _host_inputs(case, seed)
    s["case"], s["seed"] = case, seed + 17
    ctx = s["ctx"] = bm.Context(case["n"], s.pop("male"), s.pop("female"))
    ctx.set_mapping(s["pi"])
    if kind in ("table", "table3", "best"):
        ctx.gain_enable(True)
    if kind in ("table", "table3"):
        s["batch"] = ctx.batch(case["k"])
    if kind in ("learned", "mlp"):
        # He-normal weights from the seed: a network trained here would rank
        # differently from one process to the next (its gradients are summed
        # with float atomics), and which pairs lead is all the weights decide
        s["mlp"] = bm.Mlp(ctx, seed=seed)
    return s


def _counts(res):
    return {k: int(v) for k, v in res.items() if k != "seconds"}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "anneal":
        a = s["anneal"]
        a.reset()
        a.run(case["steps"], case["launches"])
        st = a.state()
        return {**st, "trajectory": a.trajectory(), "mapping": a.mapping(int(np.argmax(st["best"])), best=True)}
    ctx = s["ctx"]
    if kind == "list":
        return ctx.swap_deltas(s["uv"])
    if kind == "changed":
        return ctx.swap_deltas_changed(s["changed"])
    if kind == "changed3":
        return ctx.rot3_deltas_changed(s["changed"])
    ctx.set_mapping(s["pi"])    # the climbs and tools move it; a table is built anew
    if kind == "search":
        best, res = ctx.search(case["mode"], seed=s["seed"], max_iters=case["iters"])
        return {"best": best, "left": ctx.get_mapping(), **_counts(res)}
    if kind == "climb":
        trace, res = ctx.hillclimb(s["seed"], case["rounds"], case["batch"], verify=False)
        return {"trace": trace, "mapping": ctx.get_mapping(), **_counts(res)}
    if kind == "learned":
        trace, _, res = ctx.climb(bm.PROPOSAL_LEARNED, seed=s["seed"], max_rounds=case["rounds"],
                                  per_round=case["top"], pool=case["pool"], mlp=s["mlp"], trace_cap=case["rounds"])
        return {"trace": trace, "mapping": ctx.get_mapping(), **_counts(res)}
    if kind == "mlp":
        m = s["mlp"]
        m.set_params(s["params"])
        m.refresh_features()
        y = m.score_pairs(s["uv"])
        grad, mse = m.gradient(s["uv"], s["target"])
        losses = m.train(s["seed"], case["steps"], batch=case["k"], lr=1e-3)
        return {"y": y, "grad": grad, "mse": mse, "losses": losses, "params": m.params()}
    if kind == "best":
        trace, res = ctx.best_swap_climb(case["iters"], verify_every=0)
        return {"trace": trace, "mapping": ctx.get_mapping(), **_counts(res)}
    b = s["batch"]
    if kind == "table":
        b.eval_swaps_umajor(s["seed"], case["k"])
    else:
        b.eval_rot3_amajor(s["seed"], case["k"])
    st = b.stats()
    out = dict(st)
    if st["n_pos"] > 0:
        at = out["picked"] = b.pick(1, st["n_pos"] // 2)
        out["picked_delta"] = b.deltas(at, 1)
    if case["k"] <= WHOLE:
        out["deltas"] = b.deltas()
        if kind == "table3":
            out["perms"] = b.perms()
    return out


def _edges(case):
    return int(case["n"] * case["deg"])


def work(case):
    """Bytes and operations of one pass: each list of both graphs that the
    path needs read once (8 bytes an entry), outputs written once; one
    operation per term min(w, w_F) that has to be formed or per table entry
    combined."""
    kind, deg = case["kind"], case["deg"]
    if kind == "anneal":
        n = [int(x) for x in case["sizes"].split(",")]
        steps = len(n) * case["chains"] * case["steps"] * case["launches"]
        return {"bytes": sum(4 * x * deg * 8 + 2 * case["chains"] * 4 * x for x in n), "flops": steps * 4 * deg * 2}
    n, m = case["n"], _edges(case)
    graphs = 4 * m * 8 + 8 * n
    if kind == "list":
        touched = min(4 * m, case["k"] * 8 * deg)
        return {"bytes": 16 * case["k"] + 8 * touched, "flops": case["k"] * 8 * deg}
    if kind in ("changed", "changed3"):
        c = case["c"]
        k = n * c if kind == "changed" else n * c * (c + 1) / 2
        # a placement row and column of each changed vertex, every candidate's delta and ids
        return {"bytes": graphs + (16 if kind == "changed" else 24) * k, "flops": 8 * k + (c + 1) * 4 * deg * deg}
    if kind == "search":
        c = 200 if case["mode"] == 0 else 8
        per = n * c * (c if case["mode"] == 2 else 2) / 2 + case["iters"] * n * (6 if case["mode"] == 2 else 2)
        # a placement row and column of each changed vertex, and every candidate's delta
        return {"bytes": graphs + 8 * per, "flops": 4 * per + (c + 3 * case["iters"]) * 4 * deg * deg}
    if kind == "climb":
        k = case["rounds"] * case["batch"]
        return {"bytes": graphs + 8 * n, "flops": k * 8 * deg}
    if kind == "learned":
        return {"bytes": graphs + case["rounds"] * (32 * n + 8 * case["top"]),
                "flops": case["rounds"] * (case["pool"] * 37120 + case["top"] * 8 * deg)}
    if kind == "mlp":
        k = case["k"]
        return {"bytes": graphs + 16 * k + 8 * 18817, "flops": 37120.0 * k * (1 + 3 * (1 + case["steps"]))}
    table = 4 * n * n
    if kind == "best":
        return {"bytes": graphs + table * (2 + case["iters"]), "flops": case["iters"] * 8 * n * n / 2}
    outs = case["k"] * (9 if kind == "table3" else 8)
    return {"bytes": graphs + table + outs, "flops": 4 * m * deg + case["k"] * (30 if kind == "table3" else 6)}


# ---------------------------------------------------------------------------
# the same numbers from numpy alone


class _Pair:
    """Both graphs as sorted edge keys, for lookups."""

    def __init__(self, n, male, female):
        self.n = n
        self.female = self._last(female)
        key, w = self._last(male)
        self.mu, self.mx, self.mw = key // (n + 1), key % (n + 1), w

    def _last(self, g):
        """Edge keys ascending, the last line of each (src, dst) kept."""
        key = g.src.astype(np.int64)[::-1] * (self.n + 1) + g.dst.astype(np.int64)[::-1]
        key, at = np.unique(key, return_index=True)
        return key, g.w.astype(np.int64)[::-1][at]

    def terms(self, w, a, b):
        """min(w, w_F(a, b)) where F has the edge, else 0."""
        fk, fw = self.female
        key = a.astype(np.int64) * (self.n + 1) + b
        at = np.minimum(np.searchsorted(fk, key), len(fk) - 1)
        return np.where(fk[at] == key, np.minimum(w, fw[at]), 0)


def _exact_list(case, s, pairs):
    n, pi = case["n"], s["pi"].astype(np.int64)
    p = _Pair(n, s["male"], s["female"])
    by_out = np.searchsorted(p.mu, np.arange(n + 2))
    order = np.argsort(p.mx, kind="stable")
    by_in = np.searchsorted(p.mx[order], np.arange(n + 2))
    out = np.zeros(len(pairs), np.int64)
    for i, (u, v) in enumerate(pairs.tolist()):
        e = np.unique(np.concatenate([np.arange(by_out[u], by_out[u + 1]), np.arange(by_out[v], by_out[v + 1]),
                                      order[by_in[u]:by_in[u + 1]], order[by_in[v]:by_in[v + 1]]]))
        a, b, w = p.mu[e], p.mx[e], p.mw[e]
        qa = np.where(a == u, pi[v], np.where(a == v, pi[u], pi[a]))
        qb = np.where(b == u, pi[v], np.where(b == v, pi[u], pi[b]))
        out[i] = (p.terms(w, qa, qb) - p.terms(w, pi[a], pi[b])).sum()
    return out


def _exact_features(case, s):
    """The eight inputs per vertex (include/brainmatch.h, learned swap proposal)."""
    n, pi = case["n"], s["pi"].astype(np.int64)
    p = _Pair(n, s["male"], s["female"])
    c = p.terms(p.mw, pi[p.mu], pi[p.mx])
    count = lambda at: np.bincount(at, minlength=n + 1).astype(np.float64)  # noqa: E731
    total = lambda at, x: np.bincount(at, weights=x, minlength=n + 1)  # noqa: E731
    od, idg = count(p.mu), count(p.mx)
    wsum = total(p.mu, p.mw) + total(p.mx, p.mw)
    carried = total(p.mu, c) + total(p.mx, c)
    zero = total(p.mu, c == 0) + total(p.mx, c == 0)
    fk = p.female[0]
    fo, fi = count(fk // (n + 1)), count(fk % (n + 1))
    f = np.stack([np.log1p(od), np.log1p(idg), np.log1p(wsum), carried / (wsum + 1), zero / (od + idg + 1),
                  np.log1p(fo[pi]), np.log1p(fi[pi]), np.log1p(carried)], axis=1)
    f[0] = 0
    return f


def exact(case, seed):
    kind = case["kind"]
    if kind == "list" and case["k"] * case["deg"] <= 1.5e6:
        s = _host_inputs(case, seed)
        return _exact_list(case, s, s["uv"])
    if kind == "changed" and case["c"] * case["n"] * case["deg"] <= 1.5e6:
        s = _host_inputs(case, seed)
        first = np.sort(s["changed"])
        order = np.concatenate([first, np.setdiff1d(np.arange(1, case["n"] + 1), first)])
        pairs = np.concatenate([np.stack([np.full(case["n"] - 1 - i, u), order[i + 1:]], axis=1)
                                for i, u in enumerate(first)]).astype(np.int32)
        return _exact_list(case, s, pairs), pairs
    if kind == "mlp":
        s = _host_inputs(case, seed)
        f = _exact_features(case, s)
        q = s["params"].astype(np.float64)
        w1, b1, w2, b2, w3, b3 = np.split(q, np.cumsum([2048, 128, 16384, 128, 128]))
        w1, w2 = w1.reshape(16, 128), w2.reshape(128, 128)
        x = np.concatenate([f[s["uv"][:, 0]], f[s["uv"][:, 1]]], axis=1)
        z1 = x @ w1 + b1
        h1 = np.maximum(z1, 0)
        z2 = h1 @ w2 + b2
        h2 = np.maximum(z2, 0)
        y = h2 @ w3 + b3
        d = y - s["target"]
        dy = 2 * d / len(d)
        g2 = dy[:, None] * w3 * (z2 > 0)
        g1 = (g2 @ w2.T) * (z1 > 0)
        grad = np.concatenate([(x.T @ g1).ravel(), g1.sum(0), (h1.T @ g2).ravel(), g2.sum(0), h2.T @ dy, [dy.sum()]])
        return {"y": y, "grad": grad, "mse": float(np.mean(d * d)), "losses": None, "params": None}
    return None
