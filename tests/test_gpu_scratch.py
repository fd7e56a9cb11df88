"""Calls whose scratch memory cannot be allocated: where an older form of the
work needs none, it runs.  A child process puts its own hipMalloc in front of
the runtime's, which refuses from a given size on."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static size_t from = (size_t)-1;
static long refused_calls;
void refuse_from(size_t bytes) { from = bytes; }
long refused(void) { return refused_calls; }
int hipMalloc(void** p, size_t bytes) {
    static int (*next)(void**, size_t);
    if (!next) next = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD), "hipMalloc");
    if (bytes >= from) { refused_calls++; return 2; }   /* hipErrorOutOfMemory */
    return next(p, bytes);
}
"""

HEAD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
shim.refuse_from.argtypes = [ctypes.c_size_t]
import numpy as np
import brainmatch as bm
"""

ENUMERATIONS = r"""
n = 6000
male, female, _, pi = bm.synth_pair(n, 200.0, bm.WEIGHTS_LOGNORMAL, 0.3, seed=3)
changed = np.array([5, 17, 200, 4001, 5999], np.int32)


def both():
    with bm.Context(n, male, female) as ctx:
        ctx.set_mapping(pi)
        p, t = ctx.batch(5 * n), ctx.batch(15 * n)
        p.gen_changed_pairs(changed)
        t.gen_changed_triples(changed)
        if limit:
            shim.refuse_from(limit)
        p.eval_swaps()
        t.eval_rot3()
        out = p.deltas(), p.pairs(), t.deltas(), t.perms(), t.triples()
        shim.refuse_from(ctypes.c_size_t(-1).value)
        p.close()
        t.close()
    return out


limit = 0
want = both()
limit = 1 << 16
got = both()
assert shim.refused() >= 2, shim.refused()
for a, b in zip(want, got):
    assert np.array_equal(a, b)
print("SCRATCH_OK", flush=True)
"""


TRAINING = r"""
n = 300
male, female, _, pi = bm.synth_pair(n, 8.0, bm.WEIGHTS_GEOMETRIC, 0.3, seed=3)
with bm.Context(n, male, female) as ctx:
    ctx.set_mapping(pi)

    def losses(steps, limit):
        with bm.Mlp(ctx, seed=1) as m:
            p = m.params()
            m.train(4, 2, batch=32, lr=1e-4)     # every buffer of a step is there
            m.set_params(p)
            if limit:
                shim.refuse_from(limit)
            out = m.train(9, steps, batch=32, lr=1e-4)
            shim.refuse_from(ctypes.c_size_t(-1).value)
            return out

    got, want = losses(20000, 1 << 16), losses(5000, 0)
    assert len(got) == 20000 and np.array_equal(got[:5000], want) and np.all(np.isfinite(got)) and np.all(got > 0)
print("SCRATCH_OK", flush=True)
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    (d / "shim.c").write_text(SHIM)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(d / "shim.so"), str(d / "shim.c"), "-ldl"], check=True)
    return str(d / "shim.so")


# placement rows: enumerations go one by one; training: a step's errors need no
# memory in proportion to the steps
@pytest.mark.parametrize("code", [ENUMERATIONS, TRAINING], ids=["enumerations", "training"])
def test_runs_without_the_memory(shim, code):
    env = dict(os.environ, PYTHONPATH=os.path.join(ROOT, "brain-match_amd"))
    r = subprocess.run([sys.executable, "-c", HEAD + code, shim], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "SCRATCH_OK" in r.stdout, r.stdout + r.stderr[-2000:]
