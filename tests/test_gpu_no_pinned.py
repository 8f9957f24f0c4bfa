"""Answers come all the same where no pinned memory is left for them: small answers, small batches, the
residuals of batched PPR, large answers and uploads.  A child process runs them with a hipHostMalloc that
refuses every request of 4000 bytes or more, preloaded beside whatever is preloaded already, and compares
with the same calls made before the refusals."""
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
int refuse_from_4000, refused;
int hipHostMalloc(void** p, size_t n, unsigned flags) {
    static int (*next)(void**, size_t, unsigned);
    if (refuse_from_4000 && n >= 4000) {
        ++refused;
        return 2; /* hipErrorOutOfMemory */
    }
    if (!next) { /* the runtime that libeegraph.so has loaded, which is in no global scope */
        void* hip = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
        if (hip) next = (int (*)(void**, size_t, unsigned))dlsym(hip, "hipHostMalloc");
    }
    return next ? next(p, n, flags) : 1; /* hipErrorInvalidValue */
}
"""

CHILD = r"""
import ctypes, sys
sys.path.insert(0, sys.argv[1])
import numpy as np
import eegraph_amd as eg

shim = ctypes.CDLL(sys.argv[2])
refuse, refused = (ctypes.c_int.in_dll(shim, x) for x in ("refuse_from_4000", "refused"))

def answers(n, m):
    rng = np.random.default_rng(n)
    s, d, w = (rng.integers(lo, hi, m).astype(np.uint32) for lo, hi in ((0, n), (0, n), (1, 60)))
    with eg.Graph.from_edges(s, d, w, n=n) as g:
        print("case", n, m, "refusing" if refuse.value else "", flush=True)
        out = [g.run("sssp", 1)[0], g.run("cc", 0)[0], g.run("ppr", 1)[0]]
        out += [g.run_batch(a, np.arange(k))[0] for a, k in (("bfs", 3), ("sssp", 2), ("sssp", 20), ("ppr", 3))]
        return out

CASES = [(5000, 30000), (300_001, 900_000), (2_200_000, 2_300_000)]
want = [answers(*c) for c in CASES[:1]] + [None, None]
refuse.value = 1
got = [answers(*c) for c in CASES]
assert refused.value >= 6, refused.value
refuse.value = 0
want[1:] = [answers(*c) for c in CASES[1:]]
for a, b in zip(got, want):
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and np.array_equal(x.view(np.uint32), y.view(np.uint32))
print("same answers,", refused.value, "refusals")
"""


@pytest.mark.skipif(not shutil.which("gcc"), reason="needs gcc")
def test_without_pinned_memory(tmp_path):
    (tmp_path / "shim.c").write_text(SHIM)
    (tmp_path / "child.py").write_text(CHILD)
    so = str(tmp_path / "shim.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", str(tmp_path / "shim.c"), "-o", so, "-ldl"], check=True)
    env = dict(os.environ, LD_PRELOAD=":".join(x for x in (os.environ.get("LD_PRELOAD"), so) if x))
    r = subprocess.run([sys.executable, "-u", str(tmp_path / "child.py"), ROOT, so], env=env, capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr[-2000:]
    assert "same answers" in r.stdout
