"""Ranks are rounded once: along the chain 0 -> 1 -> 2 -> 3 a rank is base + d * c exactly (a 48-bit
product), kept as a pair, and goes out and into the next contribution as its nearest float.  The values
expected are computed in FP64 and rounded to float once; equality, since a pair holds ~46 bits and a
product within 2^-46 of the middle between two floats does not occur among these."""
import numpy as np
import pytest

import eegraph_amd as eg

pytestmark = pytest.mark.gpu

DAMPING = np.random.default_rng(5).uniform(0.3, 0.97, 64).astype(np.float32)


def chain_ranks(d, base, restart):
    """base: the teleport term of every vertex; restart: that of vertex 0."""
    x = [np.float32(restart)]
    for _ in range(3):
        x.append(np.float32(np.float64(base) + np.float64(d) * np.float64(x[-1])))
    return np.array(x, np.float32)


@pytest.fixture(scope="module")
def chain():
    with eg.Graph.from_edges([0, 1, 2], [1, 2, 3], None, n=4) as g:
        yield g


@pytest.mark.parametrize("nsrc", [1, 9, 17])  # planes of 8, 16 and 32 columns
def test_batched(chain, nsrc):
    for d in DAMPING:
        out, _ = chain.run_batch("ppr", [0] * nsrc, damping=float(d))
        want = chain_ranks(d, 0.0, np.float32(1) - d)
        for row in out:
            assert np.array_equal(row.view(np.uint32), want.view(np.uint32)), (d, row, want)


@pytest.mark.parametrize("K", [4, 8, 16, 32])
@pytest.mark.parametrize("algo", ["pr", "ppr"])
def test_in_place(chain, algo, K):
    for d in DAMPING:
        out, _ = chain.run(algo, 0, variant="async_push_dd", K=K, damping=float(d))
        base = np.float32(0) if algo == "ppr" else (np.float32(1) - d) / np.float32(4)
        want = chain_ranks(d, base, np.float32(1) - d if algo == "ppr" else base)
        assert np.array_equal(out.view(np.uint32), want.view(np.uint32)), (d, out, want)
