"""The default frontier queue on both sides of the size where its form changes (2^19 vertices): the
oracle's labels, several runs on one handle, activity summing to the same frontiers as flag scans
reach."""
import numpy as np
import pytest

import eegraph_amd as eg
import oracle_py as O

pytestmark = pytest.mark.gpu

ALG = {"bfs": O.BFS, "sssp": O.SSSP, "sswp": O.SSWP}


@pytest.mark.parametrize("n", [(1 << 19) - 1, 1 << 19])
def test_both_sides(n):
    rng = np.random.default_rng(n)
    m = 3 * n
    s, d, w = (rng.integers(lo, hi, m).astype(np.uint32) for lo, hi in ((0, n), (0, n), (1, 30)))
    with eg.Graph.from_edges(s, d, w, n=n) as g:
        for alg in ALG:
            for src in (1, n - 1, 1):
                out, st = g.run(alg, src, variant="sync_push_dd", K=8)
                assert np.array_equal(out, O.reference_labels(ALG[alg], n, s, d, w, src)), (alg, src)
        act, st = g.run("bfs", 1, variant="sync_push_dd", K=8, activity_cap=64)
        ref, sr = g.run("bfs", 1, variant="sync_push_dd", frontier="compact", K=8, activity_cap=64)
        assert np.array_equal(act, ref) and list(st["activity"]) == list(sr["activity"])
        lim, _ = g.run("cc", 0, variant="sync_push_dd", K=8, count_work=True)
        assert np.array_equal(lim, O.wcc(n, s, d))
