"""In-place PageRank where the first sweep changes nothing but the vertices without in-edges: with one
edge into and out of every other vertex, x = 1/N is a fixed point until the teleport term of the first
vertex arrives, so only that vertex's change keeps the run going.

Tolerance: the two iterations stop at the same L1 change, 1e-7, at most 1e-7 * d / (1 - d) from the
fixed point each, and ranks are single floats (2^-24): below 2e-6.
"""
import numpy as np
import pytest

import eegraph_amd as eg
import oracle_py as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", ["async_push_td", "async_push_dd"])
@pytest.mark.parametrize("n", [2, 4, 300, 5000])
def test_chain(n, variant):
    s = np.arange(n - 1, dtype=np.uint32)
    d = s + 1
    row, col, _ = O.csr(n, s, d)
    ref, _, _ = O.pagerank(n, row, col, 0.85, 1e-7)
    with eg.Graph.from_edges(s, d, None, n=n) as g:
        out, st = g.run("pr", 0, variant=variant)
    assert st["iterations"] > 1
    assert np.abs(out.astype(np.float64) - ref).sum() < 2e-6
