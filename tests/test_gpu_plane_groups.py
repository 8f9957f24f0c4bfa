"""Narrow label planes with several virtual nodes side by side in a wavefront (rows of 16 and 32
lane words): the widths where the grouping changes, on a graph whose last tiles are ragged, against
32-bit planes."""
import numpy as np
import pytest

import eegraph_amd as eg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alg,wmax,bits", [("sssp", 3, 8), ("sssp", 1000, 16), ("sswp", 200, 8)])
@pytest.mark.parametrize("n", [61, 7777])
def test_groups_equal_32_bit(alg, wmax, bits, n):
    rng = np.random.default_rng(n)
    m = 11 * n + 3
    s, d = rng.integers(0, n, m), (rng.integers(0, n, m) * rng.random(m) ** 3).astype(int)  # few hubs get most edges
    s[: m // 3] = rng.integers(0, 1 + n // 50, m // 3)  # and few have most out-edges
    w = rng.integers(1, wmax + 1, m)
    with eg.Graph.from_edges(s, d, w, n=n) as g:
        for nsrc in (17, 64, 65, 128, 129, 192, 193):
            srcs = rng.integers(0, n, nsrc).astype(np.uint32)
            for K in (4, 8, 16, 32):
                out, st = g.run_batch(alg, srcs, K=K)
                assert st["label_bits"] == bits
                ref, _ = g.run_batch(alg, srcs, K=K, label_bits=32)
                assert np.array_equal(out, ref), (nsrc, K)
