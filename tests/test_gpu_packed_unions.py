"""Packed runs on changing lists of graphs: the union's memory passes from list to list, larger and
smaller, weighted and not; members around the chunks of the copy (16384 edges and vertices)."""
import numpy as np
import pytest

import eegraph_amd as eg

pytestmark = pytest.mark.gpu


def member(n, m, weighted, seed):
    rng = np.random.default_rng(seed)
    s, d, w = (rng.integers(lo, hi, m).astype(np.uint32) for lo, hi in ((0, n), (0, n), (1, 50)))
    return eg.Graph.from_edges(s, d, w if weighted else None, n=n)


LISTS = [([(16384, 16384), (16383, 16385), (16385, 1), (1, 0), (7, 40_000)], True),
         ([(100, 300), (2, 1)], True),
         ([(60_000, 200_000), (40_000, 16_383), (3, 0)], False),
         ([(1 << 17, 1 << 20), (5, 32_768)], True)]


def test_lists_in_turn():
    lists = [([member(n, m, wt, 10 * i + j) for j, (n, m) in enumerate(sizes)], wt)
             for i, (sizes, wt) in enumerate(LISTS)]
    for i in (0, 1, 3, 2, 1, 0, 3):
        gs, weighted = lists[i]
        for alg in ("bfs", "cc") + (("sssp", "sswp") if weighted else ()):
            for kw in (dict(variant="sync_push_dd"), dict(variant="sync_push_dd", frontier="flags"),
                       dict(variant="sync_push_dd", frontier="compact"), dict(variant="async_push_dd")):
                outs, _ = eg.run_packed(gs, alg, [g.info()["n"] - 1 for g in gs], K=8, **kw)
                for g, out in zip(gs, outs):
                    assert np.array_equal(out, g.run(alg, g.info()["n"] - 1, K=8)[0]), (i, alg, kw)
    for gs, _ in lists:
        for g in gs:
            g.close()
