"""The streamed PageRank gather at the edges of its tiles: 16 edges per lane, 1024 per wave tile,
rows that end, start or continue there, and more than 8 tiles in one row.

Tolerance: the ranks' only 32-bit roundings are those of the contributions and of the result,
2^-24 each; an iteration passes on at most d = 0.85 of the error it finds, so the L1 distance to
the FP64 iteration stays below 2^-24 * (1 + 2 / (1 - d)) < 1e-6.
"""
import numpy as np
import pytest

import eegraph_amd as eg
import oracle_py as O

pytestmark = pytest.mark.gpu

L1_TOL = 1e-6


def in_degrees(indeg, n, seed):
    """An edge list with the given in-degrees (vertex i has indeg[i]), sources at random."""
    rng = np.random.default_rng(seed)
    d = np.repeat(np.arange(len(indeg), dtype=np.uint32), indeg)
    return rng.integers(0, n, len(d)).astype(np.uint32), d


@pytest.mark.parametrize("indeg", [
    [1], [15], [16], [17], [1] * 16, [1] * 1024, [1023, 1], [1024, 1], [1025, 1],
    [3] * 341 + [1, 2, 5], [1024] * 9, [8191, 1, 1], [9 * 1024, 7], [9 * 1024 + 1, 1024, 16] + [1] * 40,
    [100_003] + [2] * 5000 + [1000] * 9,
])
@pytest.mark.parametrize("algo", ["pr", "ppr"])
def test_stream_tile_edges(indeg, algo):
    n = max(len(indeg) + 3, 2000)
    s, d = in_degrees(indeg, n, 11)
    row, col, _ = O.csr(n, s, d)
    src = int(s[0])
    xo, it_o, _ = O.pagerank(n, row, col, 0.85, 1e-7, personalised=algo == "ppr", source=src)
    with eg.Graph.from_edges(s, d, None, n=n) as g:
        x, st = g.run(algo, src, variant="sync_push_dd")
    assert abs(int(st["iterations"]) - int(it_o)) <= 1
    assert np.abs(x.astype(np.float64) - xo).sum() < L1_TOL


@pytest.mark.parametrize("n", [1, 3, 4, 38911, 38912, 38913, 60000])
def test_stream_hub_table_sizes(n):
    """Vertex counts around a 4-vertex load and around the hubs that fit in LDS."""
    rng = np.random.default_rng(n)
    m = 40 * n + 1
    s, d = (rng.integers(0, n, m).astype(np.uint32) for _ in range(2))
    row, col, _ = O.csr(n, s, d)
    xo, it_o, _ = O.pagerank(n, row, col, 0.85, 1e-7)
    with eg.Graph.from_edges(s, d, None, n=n) as g:
        x, st = g.run("pr", 0, variant="sync_push_dd")
        y, _ = g.run("pr", 0, variant="sync_push_dd", wgs_per_cu=7)
    assert abs(int(st["iterations"]) - int(it_o)) <= 1
    assert np.abs(x.astype(np.float64) - xo).sum() < L1_TOL
    assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
