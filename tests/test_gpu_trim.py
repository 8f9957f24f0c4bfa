"""Memory of closed handles: kept for the next ones (bounded), given back by trim(), and given back
without it when a handle is closed on a card that is nearly full.  Free memory comes from the HIP runtime
that libeegraph.so is linked against."""
import ctypes as C

import numpy as np
import pytest

import eegraph_amd as eg

pytestmark = pytest.mark.gpu

_hip = C.CDLL("libamdhip64.so.7")
_hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
_hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
_hip.hipFree.argtypes = [C.c_void_p]
MIB = 1 << 20


def free_bytes():
    a, t = C.c_size_t(), C.c_size_t()
    assert _hip.hipMemGetInfo(C.byref(a), C.byref(t)) == 0
    return a.value, t.value


def use(scale):
    s, d, w = eg.gen_rmat(scale, 16, seed=3)
    with eg.Graph.from_edges(s, d, w, n=1 << scale) as g:
        return g.run("sssp", 1)[0], g.run("pr", 0)[0], g.run_batch("bfs", np.arange(5))[0]


def test_trim_gives_back_what_closed_handles_held():
    first = use(18)  # code objects, scratch
    eg.trim()
    before, _ = free_bytes()
    again = use(18)
    kept = before - free_bytes()[0]
    assert 0 < kept <= 1024 * MIB + 64 * MIB
    assert eg.trim() >= kept - 64 * MIB
    assert free_bytes()[0] >= before - 2 * MIB
    assert eg.trim() == 0
    for a, b, c in zip(first, again, use(18)):
        assert np.array_equal(a, b) and np.array_equal(a, c)


def test_trim_leaves_open_handles_alone():
    s, d, w = eg.gen_rmat(14, 16, seed=4)
    with eg.Graph.from_edges(s, d, w, n=1 << 14) as g:
        want = g.run("sssp", 1)[0]
        use(12)
        eg.trim()
        assert np.array_equal(g.run("sssp", 1)[0], want)


def test_closing_on_a_full_card_gives_back():
    use(18)
    eg.trim()
    avail, total = free_bytes()
    hold = C.c_void_p()
    assert _hip.hipMalloc(C.byref(hold), avail - total // 10) == 0  # a tenth is left
    try:
        before, _ = free_bytes()
        use(18)
        assert free_bytes()[0] >= before - 2 * MIB
    finally:
        _hip.hipFree(hold)
