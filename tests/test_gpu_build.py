"""Device graph construction: rows in input order with parallel edges and self-loops, weighted and
not, isolated vertices, around the sizes of the sorts' tiles and of the upload's slots."""
import numpy as np
import pytest

import eegraph_amd as eg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weighted", [True, False])
@pytest.mark.parametrize("n,m", [(1, 0), (1, 5), (2, 1), (300, 255), (65_537, 4097), (1000, 100_003),
                                 (700_001, 699_051), (70_000, 2_097_153)])
def test_rows(n, m, weighted):
    rng = np.random.default_rng(m)
    s = (rng.integers(0, n, m) * rng.random(m) ** 2).astype(np.uint32)
    d = rng.integers(0, n, m).astype(np.uint32)
    w = rng.integers(0, 1 << 32, m, dtype=np.uint64).astype(np.uint32) if weighted else None
    with eg.Graph.from_edges(s, d, w, n=n) as g:
        row, col, wgt = g.csr_export()
        irow, icol = g.csr_export_derived("in")
        info = g.info()
    order = np.argsort(s, kind="stable")
    deg = np.bincount(s, minlength=n)
    assert np.array_equal(row, np.r_[0, np.cumsum(deg)])
    assert np.array_equal(col, d[order])
    if weighted:
        assert np.array_equal(wgt, w[order])
    assert (info["max_out_degree"], info["argmax_out_degree"], info["nonzero_out"]) == \
        (deg.max(), deg.argmax(), np.count_nonzero(deg))
    assert np.array_equal(irow, np.r_[0, np.cumsum(np.bincount(d, minlength=n))])
    for v in (0, n // 2, n - 1):  # sources of an in-edge row: the same set of edges
        assert np.array_equal(np.sort(icol[int(irow[v]):int(irow[v + 1])]), np.sort(s[d == v]))


def test_endpoints_are_checked():
    for s, d in (([0, 5], [1, 1]), ([0, 1], [1, 7])):
        with pytest.raises(eg.EEGError):
            eg.Graph.from_edges(s, d, [1, 1], n=5)
