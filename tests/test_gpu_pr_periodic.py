"""PageRank where paths have a period (grids, bipartite graphs): every form of the iteration meets
its 1e-7 stop, as soon as the FP64 iteration does, and holds the right ranks.  Sizes lie on both sides of
the 19,456 vertices up to which single queries carry contributions as pairs.

Tolerance against the FP64 iteration run to 1e-12: stopping at an L1 change of 1e-7 leaves at most
1e-7 * d / (1 - d); contributions are off by at most 2^-23 (their rounding and the last one's, fed back),
of which an iteration passes on d, and the result is rounded to 2^-24:
1e-7 * d / (1 - d) + 2^-24 * (1 + 2 / (1 - d)) < 1.5e-6 at d = 0.85.
"""
import numpy as np
import pytest

import eegraph_amd as eg
import oracle_py as O

pytestmark = pytest.mark.gpu

L1_TOL = 1.5e-6


def bipartite(a, b, m, seed):
    rng = np.random.default_rng(seed)
    u, v = rng.integers(0, a, m).astype(np.uint32), (a + rng.integers(0, b, m)).astype(np.uint32)
    return a + b, np.r_[u, v], np.r_[v, u]


def grid(w, h):
    s, d, _ = eg.gen_grid(w, h, 0.01, seed=3, wmin=1, wmax=1)
    return w * h, s, d


GRAPHS = {"grid-47x297": lambda: grid(47, 297), "grid-300x200": lambda: grid(300, 200),
          "bipartite-3-20000": lambda: bipartite(3, 20000, 30000, 1),
          "bipartite-1-25000": lambda: bipartite(1, 25000, 60000, 2),
          "bipartite-2000-20000": lambda: bipartite(2000, 20000, 60000, 3)}
GRAPHS.update({f"bipartite-small-{k}": (lambda k=k: bipartite(1 + k % 5, 2 + k % 4, 3 + 5 * k, k)) for k in range(8)})


@pytest.fixture(scope="module", params=list(GRAPHS))
def case(request):
    n, s, d = GRAPHS[request.param]()
    row, col, _ = O.csr(n, s, d)
    srcs = np.unique(np.r_[s[0], d[0], np.random.default_rng(n).choice(s, 15)]).astype(np.uint32)

    def ref(algo, src=0):
        args = dict(personalised=algo == "ppr", source=int(src))
        x, _, _ = O.pagerank(n, row, col, 0.85, 1e-12, **args)
        return x, O.pagerank(n, row, col, 0.85, 1e-7, **args)[1]

    with eg.Graph.from_edges(s, d, None, n=n) as g:
        yield n, g, srcs, ref, [ref("ppr", x) for x in srcs]


def check(x, iterations, ref):
    assert np.abs(x.astype(np.float64) - ref[0]).sum() < L1_TOL
    assert iterations <= 2 * ref[1]


def test_single(case):
    n, g, srcs, ref, ppr = case
    x, st = g.run("pr", 0, variant="sync_push_dd")
    check(x, st["iterations"], ref("pr"))
    for src, r in zip(srcs[:4], ppr):
        x, st = g.run("ppr", int(src), variant="sync_push_dd")
        check(x, st["iterations"], r)


def test_in_place(case):
    n, g, srcs, ref, ppr = case
    x, st = g.run("pr", 0, variant="async_push_dd")
    check(x, st["iterations"], ref("pr"))
    for src, r in zip(srcs[:6], ppr):
        x, st = g.run("ppr", int(src), variant="async_push_dd")
        check(x, st["iterations"], r)


@pytest.mark.parametrize("nsrc", [5, 9, 40])  # planes of 8, 16 and 32 columns, and columns taken over
def test_batched(case, nsrc):
    n, g, srcs, ref, ppr = case
    pick = np.arange(nsrc) % len(srcs)
    x, st = g.run_batch("ppr", srcs[pick])
    for row, k in zip(x, pick):
        check(row, st["iterations"], (ppr[k][0], max(r[1] for r in ppr)))


def test_served(case):
    n, g, srcs, ref, ppr = case
    with eg.Server(g, K=8) as srv:
        pick = np.arange(24) % len(srcs)
        for t, k in [(srv.submit("ppr", int(srcs[k])), k) for k in pick]:
            x, _ = srv.wait(t, algo="ppr")
            check(x, 0, ppr[k])
