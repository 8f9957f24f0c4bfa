"""Components where first edges form long chains: wheels and paths in both directions, around the steps
that a chain is walked (128) and the threads of a wave, and past what runs at once.  The time: a chain of
2^22 vertices beside a common neighbour took 162 ms when it was walked step by step, and takes 0.8."""
import numpy as np
import pytest

import eegraph_amd as eg
import oracle_py as O

pytestmark = pytest.mark.gpu


def wheel(n, rim_first=True, down=True):
    v = np.arange(1, n - 1, dtype=np.uint32)
    rim, spokes = (v, v + 1), (np.zeros(n - 1, np.uint32), np.arange(1, n, dtype=np.uint32))
    parts = (rim, spokes) if rim_first else (spokes, rim)
    s, d = (np.concatenate(x) for x in zip(*parts))
    return (d, s) if down else (s, d)


@pytest.mark.parametrize("n", [3, 64, 127, 128, 129, 130, 131, 257, 4099, 300_001])
@pytest.mark.parametrize("sym", [False, True])
def test_labels(n, sym):
    v = np.arange(n - 1, dtype=np.uint32)
    shuffled = np.random.default_rng(n).permutation(n).astype(np.uint32)
    graphs = [wheel(n, a, b) for a in (True, False) for b in (True, False)]
    graphs += [(v, v + 1), (v + 1, v), (shuffled[:-1], shuffled[1:])]
    cut = np.arange(n - 1) % 1000 != 700  # several chains
    graphs += [(s[:n - 1][cut], d[:n - 1][cut]) for s, d in graphs[4:]]
    for k, (s, d) in enumerate(graphs):
        with eg.Graph.from_edges(s, d, None, n=n) as g:
            if sym:
                g.prepare(8, eg._lib.PREP_SYM)
            out, _ = g.run("cc", 0)
        assert np.array_equal(out, O.wcc(n, s, d)), k


@pytest.mark.parametrize("sym", [False, True])
@pytest.mark.parametrize("leaves", [1, 2, 3, 4, 65, 66, 67, 129, 1000])
def test_forests(leaves, sym):
    """Beside a giant component, trees whose hubs have around the two edges that are linked first, and the
    64 more that a wave takes at once; joined in pairs by their last leaves."""
    rng = np.random.default_rng(leaves)
    k, giant = 40, 5000
    hubs = giant + (leaves + 1) * np.arange(k)
    s = np.r_[rng.integers(0, giant, 4 * giant), np.repeat(hubs, leaves), (hubs + leaves)[::2]]
    d = np.r_[rng.integers(0, giant, 4 * giant), (hubs[:, None] + np.arange(1, leaves + 1)).ravel(), (hubs + leaves)[1::2]]
    n = giant + (leaves + 1) * k
    ids = rng.permutation(n)
    s, d = (ids[x].astype(np.uint32) for x in (s, d))
    with eg.Graph.from_edges(s, d, None, n=n) as g:
        if sym:
            g.prepare(8, eg._lib.PREP_SYM)
        assert np.array_equal(g.run("cc", 0)[0], O.wcc(n, s, d))


def test_long_chains_take_no_long_time():
    n = 1 << 22
    s, d = wheel(n)
    with eg.Graph.from_edges(s, d, None, n=n) as g:
        runs = [g.run("cc", 0) for _ in range(3)]
    assert all(not out.any() for out, _ in runs)
    assert min(st["ms_traversal"] for _, st in runs) < 10
