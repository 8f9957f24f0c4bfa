"""Iteration limits: how many iterations a limit admits (whole chunks: 1 + 6 k of a queue; 6 + 8 k with
every launch timed; batched levels rounded up to 6, or 8 with timing), and that a handle whose run was
stopped answers the next one as if nothing had been.

Along the path 0 -> 1 -> .. -> L a BFS from 0 takes L iterations and one more that finds nothing."""
import ctypes as C

import numpy as np
import pytest

import eegraph_amd as eg
import eegraph_amd._lib as L
import oracle_py as O

pytestmark = pytest.mark.gpu

SIZES = [64, (1 << 19) + 13]  # pushed and sorted default queues


def path(n, length):
    s = np.arange(length, dtype=np.uint32)
    return eg.Graph.from_edges(s, s + 1, np.full(length, 3, np.uint32), n=n)


def converges(run):
    try:
        run()
        return True
    except eg.EEGError as e:
        assert "not converged" in str(e)
        return False


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("max_iters,timing,limit", [(1, False, 7), (7, False, 7), (8, False, 13), (13, False, 13),
                                                    (14, False, 19), (1, True, 6), (6, True, 6), (7, True, 14),
                                                    (8, True, 14), (14, True, 14), (15, True, 22)])
def test_admitted_iterations(n, max_iters, timing, limit):
    for length, ok in ((limit - 1, True), (limit, False)):
        with path(n, length) as g:
            for alg in ("bfs", "sssp"):
                for frontier in ("sorted", "compact"):
                    assert ok == converges(lambda: g.run(alg, 0, variant="sync_push_dd", frontier=frontier,
                                                         max_iters=max_iters, timing=timing)), (alg, frontier)


@pytest.mark.parametrize("alg,nsrc", [("bfs", 1), ("sssp", 2), ("sssp", 20)])
@pytest.mark.parametrize("max_iters,timing,limit", [(1, False, 18), (2, False, 18), (3, False, 24), (1, True, 24),
                                                    (8, True, 24), (9, True, 32)])
def test_admitted_levels_of_a_batch(alg, nsrc, max_iters, timing, limit):
    for length, ok in ((limit - 1, True), (limit, False)):
        with path(64, length) as g:
            assert ok == converges(lambda: g.run_batch(alg, [0] * nsrc, max_iters=max_iters, timing=timing,
                                                       label_bits=32 if nsrc > 16 else 0))


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("variant,frontier", [("sync_push_dd", "sorted"), ("sync_push_dd", "compact"),
                                              ("sync_push_dd", "flags"), ("async_push_dd", "sorted"),
                                              ("sync_push_td", "sorted")])
def test_a_stopped_handle_answers_again(n, variant, frontier):
    # paths that no sweep runs through at once (their ids are shuffled), and edges beside them
    rng = np.random.default_rng(n)
    ids = rng.permutation(n).astype(np.uint32)
    length = min(n, 600)
    s = np.r_[ids[:length - 1], rng.integers(0, n, n // 2).astype(np.uint32)]
    d = np.r_[ids[1:length], rng.integers(0, n, n // 2).astype(np.uint32)]
    w = rng.integers(1, 9, len(s)).astype(np.uint32)
    src = int(ids[0])
    with eg.Graph.from_edges(s, d, w, n=n) as g:
        for alg, code in (("bfs", O.BFS), ("sssp", O.SSSP), ("sswp", O.SSWP)):
            ref = O.reference_labels(code, n, s, d, w, src)
            for max_iters in (1, 2, 5):
                converges(lambda: g.run(alg, src, variant=variant, frontier=frontier, max_iters=max_iters))
                out, _ = g.run(alg, src, variant=variant, frontier=frontier)
                assert np.array_equal(out, ref), (alg, max_iters)
                if n < 100:
                    break


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("variant,frontier,activity", [("sync_push_dd", "sorted", 0), ("sync_push_dd", "compact", 1),
                                                       ("sync_push_dd", "flags", 0), ("sync_push_dd", "sorted", 1)])
def test_a_stopped_run_reports_its_time(n, variant, frontier, activity):
    with path(n, 40) as g:
        out, st = np.empty(n, np.uint32), L.Stats()
        o = eg.make_opts(variant=variant, frontier=frontier, max_iters=3, collect_activity=bool(activity))
        rc = L.lib.eeg_run(g.handle, L.BFS, 0, C.byref(o), out.ctypes.data, C.byref(st))
        assert rc == L.ERR_NOT_CONVERGED
        assert 0 < st.ms_traversal <= st.ms_total
        assert out[0] == 0 and out[3] == 3 and out[39] == eg.DIST_INFINITY
