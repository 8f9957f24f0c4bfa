"""Union-find components against the oracle's union-find, with and without the symmetrised list,
on the shapes that the sampling, the giant component and the queue of the rest depend on."""
import numpy as np
import pytest

import eegraph_amd as eg
import oracle_py as O

pytestmark = pytest.mark.gpu


def path(n, seed=None):
    ids = np.arange(n) if seed is None else np.random.default_rng(seed).permutation(n)
    return ids[:-1], ids[1:]


def shape(name):
    rng = np.random.default_rng(5)
    if name == "one_edge":
        return 3, [2], [1]
    if name == "self_loops":
        return 100, np.arange(100), np.arange(100)
    if name == "path":
        return 20_000, *path(20_000)
    if name == "reversed_path":
        s, d = path(20_000)
        return 20_000, d[::-1], s[::-1]
    if name == "shuffled_path":
        return 30_000, *path(30_000, seed=1)
    if name == "two_stars":  # the second hub's edges all lie outside the giant component
        return 70_000, np.r_[np.zeros(40_000, int), np.full(29_000, 69_999)], np.r_[1:40_001, 40_500:69_500]
    if name == "in_star":  # every edge ends at the hub: no vertex but the leaves has out-edges
        return 5000, np.arange(1, 5000), np.zeros(4999, int)
    if name == "pairs":  # no giant component: everything goes through the queue
        return 10_000, np.arange(0, 10_000, 2), np.arange(1, 10_000, 2)
    if name == "triangles":
        a = np.arange(0, 9999, 3)
        return 9999, np.r_[a, a + 1, a + 2], np.r_[a + 1, a + 2, a]
    if name == "sparse":  # around the threshold of a giant component
        return 50_000, rng.integers(0, 50_000, 27_000), rng.integers(0, 50_000, 27_000)
    if name == "blocks_of_64":
        s = rng.integers(0, 64, 4000) + 64 * rng.integers(0, 129, 4000)
        return 64 * 129 + 1, s, s // 64 * 64 + rng.integers(0, 64, 4000)
    if name == "chunk_edges":  # 2048 edges per workgroup, one more and one less
        return 3000, rng.integers(0, 3000, 2049), rng.integers(0, 3000, 2049)
    assert name == "rmat"
    s, d, _ = eg.gen_rmat(15, 3, seed=8, weights=False)
    return 1 << 15, s, d


@pytest.mark.parametrize("prepared", [False, True], ids=["edges", "symmetrised"])
@pytest.mark.parametrize("name", ["one_edge", "self_loops", "path", "reversed_path", "shuffled_path", "two_stars",
                                  "in_star", "pairs", "triangles", "sparse", "blocks_of_64", "chunk_edges", "rmat"])
def test_components(name, prepared):
    n, s, d = shape(name)
    s, d = np.asarray(s, np.uint32), np.asarray(d, np.uint32)
    ref = O.reference_labels(O.CC, n, s, d, None, 0)
    with eg.Graph.from_edges(s, d, None, n=n) as g:
        if prepared:
            g.prepare(K=8, what=eg._lib.PREP_SYM | eg._lib.PREP_TIGR)
        for variant in ("sync_push_dd", "async_push_dd"):
            lab, st = g.run("cc", variant=variant)
            assert np.array_equal(lab, ref), variant
        lab, _ = g.run("cc", frontier="compact")  # label propagation
        assert np.array_equal(lab, ref)
