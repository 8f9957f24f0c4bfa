"""Large answers to host memory (pinned slots, copying threads): sizes around the slots, the tiles
of 64 x 64 and the shares of the threads, each label width, against the oracle."""
import numpy as np
import pytest

import eegraph_amd as eg
import oracle_py as O

pytestmark = pytest.mark.gpu

ALG = {"bfs": O.BFS, "sssp": O.SSSP, "sswp": O.SSWP}


def graph(n, wmax, seed=3):
    rng = np.random.default_rng(seed)
    m = 3 * n
    s, d, w = (rng.integers(lo, hi, m).astype(np.uint32) for lo, hi in ((0, n), (0, n), (1, wmax + 1)))
    return s, d, w


# one row of a word over four slots; fewer rows than threads; narrow labels of 8 and 16 bits and
# their last tile; a share of rows that no thread count divides; a row of fewer words than a slot's part
@pytest.mark.parametrize("alg,n,nsrc,wmax", [
    ("bfs", (1 << 21) + 1, 1, 9), ("sssp", 700_001, 3, 9), ("sssp", 131_073, 17, 9), ("sssp", 65_599, 65, 1000),
    ("sswp", 32_769, 129, 200), ("sswp", 40_001, 130, 4000), ("bfs", 8_257, 256, 9), ("bfs", 8_192, 255, 9)])
def test_batch_rows(alg, n, nsrc, wmax):
    s, d, w = graph(n, wmax)
    srcs = np.random.default_rng(nsrc).integers(0, n, nsrc).astype(np.uint32)
    with eg.Graph.from_edges(s, d, w, n=n) as g:
        out, _ = g.run_batch(alg, srcs, K=8)
        for q in sorted({0, nsrc // 2, nsrc - 1}):
            assert np.array_equal(out[q], O.reference_labels(ALG[alg], n, s, d, w, int(srcs[q]))), q
        for q in range(0, nsrc, 16):
            assert np.array_equal(out[q], g.run(alg, int(srcs[q]), K=8)[0]), q


@pytest.mark.parametrize("n", [(1 << 21) - 1, 1 << 21, (1 << 22) + 5])
def test_single_query(n):
    s, d, w = graph(n, 9)
    with eg.Graph.from_edges(s, d, w, n=n) as g:
        out, _ = g.run("sssp", 1, variant="sync_push_dd", K=8)
    assert np.array_equal(out, O.reference_labels(O.SSSP, n, s, d, w, 1))


@pytest.mark.parametrize("alg", ["bfs", "cc"])
def test_packed_bounds(alg):
    sizes = [1, 524_287, 2, 524_288, 1_500_000, 3, 700_001]  # graphs that end at, before and after slots
    gs = [graph(n, 9, seed=n) if n > 3 else (np.array([0], np.uint32), np.array([n - 1], np.uint32),
                                             np.array([1], np.uint32)) for n in sizes]
    handles = [eg.Graph.from_edges(s, d, w, n=n) for n, (s, d, w) in zip(sizes, gs)]
    outs, _ = eg.run_packed(handles, alg, [0] * len(sizes), K=8)
    for n, (s, d, w), g, out in zip(sizes, gs, handles, outs):
        assert np.array_equal(out, g.run(alg, 0, variant="sync_push_dd", K=8)[0]), n
        g.close()
