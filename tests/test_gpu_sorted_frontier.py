"""Sorted queues where they are used (2^19 vertices and more; smaller graphs run the pushed queue for
them): the oracle's labels, and the iterations, relaxed edges and frontier sizes of the pushed queue, for
every K, other grids and timed launches, run after run on one handle whose marks stay."""
import numpy as np
import pytest

import eegraph_amd as eg
import oracle_py as O

pytestmark = pytest.mark.gpu

ALG = {"bfs": O.BFS, "sssp": O.SSSP, "sswp": O.SSWP}
N = (1 << 19) + 13  # the last chunk of marks is partial, and so is its last word


@pytest.fixture(scope="module")
def case():
    rng = np.random.default_rng(8)
    m = 4 * N
    # hubs as in RMAT, isolated vertices, and a path that many iterations with thin frontiers follow
    s = (N * rng.random(m) ** 3).astype(np.uint32)
    d = rng.integers(0, N - 1000, m).astype(np.uint32)
    p = np.arange(N - 1000, N - 900, dtype=np.uint32)
    s, d = np.r_[s, s[:1], p[:-1], p[-1:]], np.r_[d, p[:1], p[1:], np.uint32([N - 1])]
    w = rng.integers(1, 50, len(s)).astype(np.uint32)
    src = int(s[0])
    refs = {a: O.reference_labels(c, N, s, d, w, src) for a, c in ALG.items()}
    refs["cc"] = O.wcc(N, s, d)
    with eg.Graph.from_edges(s, d, w, n=N) as g:
        yield g, src, refs


@pytest.mark.parametrize("K", [4, 8, 16, 32])
@pytest.mark.parametrize("alg", ["bfs", "sssp", "sswp", "cc"])
def test_against_the_pushed_queue(case, alg, K):
    g, src, refs = case
    out, st = g.run(alg, src, K=K, frontier="sorted", count_work=True)
    assert np.array_equal(out, refs[alg])
    if alg == "bfs":  # levels: every queue holds one level's vertices
        _, act = g.run(alg, src, K=K, frontier="sorted", activity_cap=4096)
        ref, pushed = g.run(alg, src, K=K, frontier="compact", activity_cap=4096, count_work=True)
        assert np.array_equal(ref, refs[alg])
        assert st["iterations"] == pushed["iterations"] > 90
        assert st["edges_relaxed"] == pushed["edges_relaxed"]
        assert np.array_equal(act["activity"], pushed["activity"])
    for wgs in (1, 7):
        out, _ = g.run(alg, src, K=K, frontier="sorted", wgs_per_cu=wgs, timing=True)
        assert np.array_equal(out, refs[alg]), wgs
    out, _ = g.run(alg, src, K=K, frontier="sorted")
    assert np.array_equal(out, refs[alg])
