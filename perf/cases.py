"""What a user of eegraph_amd has it do, as cases that a timer can run.

A case is one call (or one short session) through the package's public entry points:
  query   one traversal or PageRank on a graph handle that the program keeps (`Graph.run` with
          the answer in host memory, or `eeg_run_device` with the answer in a torch tensor)
  batch   many sources at once on a kept handle (`Graph.run_batch`)
  packed  many graphs at once, one source each (`run_packed`)
  build   the whole of a one-shot program: edge list -> handle -> one query -> handle freed
  serve   a burst of mixed queries through a running `Server`
The graphs are the repository's own kinds: RMAT (a, b, c = 0.57, 0.19, 0.19; ids folded into n
where n is no power of two) and the 4-neighbour grid with 1% shortcuts; sizes are those of its
configurations, tests and benchmark, up to what one second of preparation allows.
"""
import ctypes
import math

import numpy as np
import torch

import eegraph_amd as eg
from eegraph_amd import _lib as L

DEVICE = "cuda:0"
DAMPING = float(np.float32(0.85))  # the option is a C float
EPSILON = 1e-7
# Iterations that the L1 stop at EPSILON takes on these graphs (58 .. 67); only for work().
PR_SWEEPS = 60


def listed():
    return [
        # the smallest ordinary call: one query of the RMAT-14 parity workload, answer to the host
        {"name": "sssp_rmat14", "kind": "query", "graph": "rmat", "n": 1 << 14, "m": 16 << 14, "wmax": 64,
         "algo": "sssp", "variant": "sync_push_dd", "K": 8, "out": "host"},
        # the benchmark's RMAT-22 queries: a breadth-first search feeding a device pipeline
        {"name": "bfs_rmat22", "kind": "query", "graph": "rmat", "n": 1 << 22, "m": 16 << 22, "wmax": 64,
         "algo": "bfs", "variant": "sync_push_dd", "K": 8, "out": "device"},
        # ... the in-place variant, the other one that the benchmark times, on weighted edges
        {"name": "sswp_rmat22_async", "kind": "query", "graph": "rmat", "n": 1 << 22, "m": 16 << 22, "wmax": 64,
         "algo": "sswp", "variant": "async_push_dd", "K": 8, "out": "device"},
        # ... components of the symmetrised graph: every vertex starts active
        {"name": "cc_rmat22", "kind": "query", "graph": "rmat", "n": 1 << 22, "m": 16 << 22, "wmax": 64,
         "algo": "cc", "variant": "sync_push_dd", "K": 8, "out": "device"},
        # ... and PageRank, most of the benchmark step's time
        {"name": "pr_rmat22", "kind": "query", "graph": "rmat", "n": 1 << 22, "m": 16 << 22, "wmax": 64,
         "algo": "pr", "variant": "sync_push_dd", "K": 8, "out": "device"},
        # road-like graph: long paths, thin frontiers, many iterations (weights 1..1000)
        {"name": "sssp_grid4096", "kind": "query", "graph": "grid", "width": 4096, "height": 4096, "wmax": 1000,
         "algo": "sssp", "variant": "sync_push_dd", "K": 8, "out": "device"},
        # ragged sizes, the general form of a loaded edge list, answer to the host
        {"name": "ppr_ragged", "kind": "query", "graph": "rmat", "n": 777_777, "m": 9_876_543, "wmax": 64,
         "algo": "ppr", "variant": "sync_push_dd", "K": 8, "out": "host"},
        # batches whose answers a program reads: as many rows as fit a quarter GiB
        {"name": "bfs_batch256", "kind": "batch", "graph": "rmat", "n": 1 << 18, "m": 16 << 18, "wmax": 64,
         "algo": "bfs", "nsrc": 256, "K": 8},
        {"name": "sssp_batch64", "kind": "batch", "graph": "rmat", "n": 1 << 20, "m": 16 << 20, "wmax": 64,
         "algo": "sssp", "nsrc": 64, "K": 8},
        # the packed workload of the benchmark: 64 graphs of 2^12 .. 2^20 vertices, degree 8 .. 32
        {"name": "bfs_packed64", "kind": "packed", "graphs": 64, "lo": 12, "hi": 20, "wmax": 64,
         "algo": "bfs", "K": 8},
        # the command-line programs: edge list in host memory, one query, done
        {"name": "build_sssp_rmat20", "kind": "build", "graph": "rmat", "n": 1 << 20, "m": 16 << 20, "wmax": 64,
         "algo": "sssp", "variant": "sync_push_dd", "K": 8},
        # a burst of the serving mix (40/30/20/10 BFS/SSSP/SSWP/PPR), answers read in order
        {"name": "serve_rmat18", "kind": "serve", "graph": "rmat", "n": 1 << 18, "m": 16 << 18, "wmax": 64,
         "queries": 60, "K": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _graph(rng, most, algo):
    """A graph of at most `most` vertices (and 16 x most edges), odd sizes among them.  No grid
    for components (it has one), and no unit weights for widest paths (all alike)."""
    if algo != "cc" and rng.random() < 0.2:
        side = int(math.isqrt(most))
        w = _log_int(rng, 24, side)
        return {"graph": "grid", "width": w, "height": _log_int(rng, 24, side), "wmax": rng.choice([64, 1000])}
    n = _log_int(rng, 1 << 10, most)
    return {"graph": "rmat", "n": n, "m": int(n * rng.uniform(3, 16)), "wmax": rng.choice([1, 64, 64, 200, 1000] if algo != "sswp" else [64, 64, 200, 1000])}


def draw(rng):
    kind = rng.choice(["query"] * 6 + ["batch"] * 3 + ["packed", "build", "serve"])
    k = rng.choice([8, 8, 8, 4, 16, 32])
    if kind == "query":
        algo = rng.choice(["bfs", "sssp", "sswp", "cc", "pr", "ppr"])
        variant = "sync_push_dd" if algo in ("pr", "ppr") else rng.choice(["sync_push_dd", "sync_push_dd", "async_push_dd"])
        return dict(_graph(rng, 1 << 22, algo), kind=kind, algo=algo, variant=variant, K=k, out=rng.choice(["host", "device"]))
    if kind == "batch":
        algo = rng.choice(["bfs", "sssp", "sswp", "ppr"])
        nsrc = rng.randint(1, 32) if algo == "ppr" else _log_int(rng, 1, 256)
        return dict(_graph(rng, min(1 << 20, (1 << 26) // nsrc), algo), kind=kind, algo=algo, nsrc=nsrc, K=k)
    if kind == "packed":
        lo = rng.randint(8, 14)
        return {"kind": kind, "graphs": rng.randint(2, 64), "lo": lo, "hi": rng.randint(lo, 17), "wmax": 64,
                "algo": rng.choice(["bfs", "sssp", "sswp", "cc"]), "K": k}
    if kind == "build":
        algo = rng.choice(["bfs", "sssp", "cc", "pr"])
        return dict(_graph(rng, 1 << 20, algo), kind=kind, algo=algo, variant="sync_push_dd", K=k)
    return dict(_graph(rng, 1 << 18, "sswp"), kind=kind, queries=rng.randint(4, 60), K=8)


# ---------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _rmat(n, m, wmax, seed):
    """RMAT edges by recursive quadrants, one random number per level and edge."""
    gen = _generator(seed)
    src = torch.zeros(m, dtype=torch.int32, device=DEVICE)
    dst = torch.zeros(m, dtype=torch.int32, device=DEVICE)
    for _ in range(max(1, (n - 1).bit_length())):
        r = torch.rand(m, generator=gen, device=DEVICE)
        low = r >= 0.76
        src.mul_(2).add_(low)
        dst.mul_(2).add_(((r >= 0.57) & ~low) | (r >= 0.95))
    if n & (n - 1):
        src.remainder_(n)
        dst.remainder_(n)
    w = torch.randint(1, wmax + 1, (m,), generator=gen, device=DEVICE, dtype=torch.int32)
    return n, src, dst, w


def _grid(width, height, wmax, seed):
    """4-neighbour grid, both directions, and shortcut pairs for 1% of its undirected edges."""
    gen = _generator(seed)
    n = width * height
    ids = torch.arange(n, dtype=torch.int32, device=DEVICE).view(height, width)
    a = torch.cat([ids[:, :-1].reshape(-1), ids[:-1, :].reshape(-1)])
    b = torch.cat([ids[:, 1:].reshape(-1), ids[1:, :].reshape(-1)])
    s = torch.randint(0, n, (2, a.numel() // 100), generator=gen, device=DEVICE, dtype=torch.int32)
    src = torch.cat([a, b, s[0], s[1]])
    dst = torch.cat([b, a, s[1], s[0]])
    w = torch.randint(1, wmax + 1, (src.numel(),), generator=gen, device=DEVICE, dtype=torch.int32)
    return n, src, dst, w


def _edges(case, seed):
    if case["graph"] == "grid":
        return _grid(case["width"], case["height"], case["wmax"], seed)
    return _rmat(case["n"], case["m"], case["wmax"], seed)


def _handle(edges):
    n, src, dst, w = edges
    torch.cuda.synchronize()  # the library builds on a stream of its own
    return eg.Graph.from_device_edges(src.data_ptr(), dst.data_ptr(), w.data_ptr(), src.numel(), n)


def _tables(algo):
    return L.PREP_TIGR | {"cc": L.PREP_SYM, "pr": L.PREP_TRANSPOSE, "ppr": L.PREP_TRANSPOSE}.get(algo, 0)


def _packed_shapes(case):
    rng = np.random.default_rng([case["graphs"], case["lo"], case["hi"]])
    return [(int(s), int(e)) for s, e in zip(rng.integers(case["lo"], case["hi"] + 1, case["graphs"]),
                                             rng.integers(8, 33, case["graphs"]))]


def _sources(case, seed, n):
    return np.random.default_rng(seed).integers(0, n, case["nsrc"], dtype=np.uint32)


def _stream(case, seed, n, hub):
    """The queries of a served burst; every tenth one starts at the largest hub."""
    mix = np.random.default_rng(case["queries"])
    algos = mix.choice(["bfs", "sssp", "sswp", "ppr"], case["queries"], p=[0.4, 0.3, 0.2, 0.1])
    srcs = np.random.default_rng(seed).integers(0, n, case["queries"])
    srcs[::10] = hub
    return [(str(a), int(s)) for a, s in zip(algos, srcs)]


def prepare(case, seed):
    kind = case["kind"]
    state = dict(case)
    if kind == "packed":
        state["handles"] = [_handle(_rmat(1 << s, e << s, case["wmax"], seed * 64 + i))
                            for i, (s, e) in enumerate(_packed_shapes(case))]
        for g in state["handles"]:
            g.prepare(K=case["K"], what=_tables(case["algo"]))
        state["sources"] = [g.info()["argmax_out_degree"] for g in state["handles"]]
        return state
    edges = _edges(case, seed)
    if kind == "build":
        n, src, dst, w = edges
        state["edges"] = (n, *(x.cpu().numpy().view(np.uint32) for x in (src, dst, w)))
        return state
    g = state["handle"] = _handle(edges)
    n, hub = edges[0], g.info()["argmax_out_degree"]
    if kind == "serve":
        g.prepare(K=case["K"], what=L.PREP_TIGR | L.PREP_TRANSPOSE)
        state["server"] = eg.Server(g, K=case["K"])
        state["stream"] = _stream(case, seed, n, hub)
        return state
    g.prepare(K=case["K"], what=_tables(case["algo"]))
    if kind == "batch":
        state["sources"] = _sources(case, seed, n)
        return state
    state["source"] = hub
    if case["out"] == "device":
        state["opts"] = eg.make_opts(variant=case["variant"], K=case["K"])
        real = case["algo"] in ("pr", "ppr")
        state["labels"] = torch.empty(n, dtype=torch.float32 if real else torch.int32, device=DEVICE)
        torch.cuda.synchronize()
    return state


# ---------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind == "query" and state["out"] == "device":
        L.check(L.lib.eeg_run_device(state["handle"].handle, L.ALGOS[state["algo"]], state["source"],
                                     ctypes.byref(state["opts"]), state["labels"].data_ptr(), None, None),
                "eeg_run_device")
        return state["labels"]
    if kind == "query":
        return state["handle"].run(state["algo"], state["source"], variant=state["variant"], K=state["K"])[0]
    if kind == "batch":
        return state["handle"].run_batch(state["algo"], state["sources"], K=state["K"])[0]
    if kind == "packed":
        return eg.run_packed(state["handles"], state["algo"], state["sources"], K=state["K"])[0]
    if kind == "build":
        n, src, dst, w = state["edges"]
        with eg.Graph.from_edges(src, dst, w, n=n) as g:
            return g.run(state["algo"], g.info()["argmax_out_degree"], variant=state["variant"], K=state["K"])[0]
    srv = state["server"]
    tickets = [(srv.submit(a, s), a) for a, s in state["stream"]]
    return [srv.wait(t, algo=a)[0] for t, a in tickets]


# ---------------------------------------------------------------- the least work of a pass
def work(case):
    """Edges (and weights) and row offsets read once, answers written once; PageRank reads its
    in-edges and ranks once per sweep.  One operation per edge and query (two for PageRank)."""
    if case["kind"] == "packed":
        shapes = _packed_shapes(case)
        n, m = sum(1 << s for s, _ in shapes), sum(e << s for s, e in shapes)
    elif case["graph"] == "grid":
        n = case["width"] * case["height"]
        m = int(2 * (2 * n - case["width"] - case["height"]) * 1.01)
    else:
        n, m = case["n"], case["m"]

    def one(algo, queries):
        if algo in ("pr", "ppr"):
            return PR_SWEEPS * (4 * m + 8 * n) + 4 * n * queries, 2 * PR_SWEEPS * m * queries
        edge = {"bfs": 4, "cc": 8}.get(algo, 8)
        return edge * m + 4 * n + 4 * n * queries, m * queries

    if case["kind"] == "serve":
        share = {"bfs": 0.4, "sssp": 0.3, "sswp": 0.2, "ppr": 0.1}
        parts = [one(a, max(1, round(case["queries"] * p))) for a, p in share.items()]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    b, f = one(case["algo"], case.get("nsrc", 1))
    if case["kind"] == "build":
        b += 12 * m  # the edge list itself
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------- the answers in 64 bits
def _pagerank64(n, src, dst, seeds):
    """Columns of ranks in float64, one per restart vertex (or the uniform one for None): the
    Jacobi iteration of the operator, each column stopped by its own L1 change."""
    src, dst = src.long(), dst.long()
    deg = torch.bincount(src, minlength=n).double()
    inv = torch.where(deg > 0, 1.0 / deg, torch.zeros_like(deg))
    cols = []
    for b in range(0, len(seeds), 4):
        part = seeds[b:b + 4]
        restart = torch.zeros(n, len(part), dtype=torch.float64, device=DEVICE)
        for q, s in enumerate(part):
            if s is None:
                restart[:, q] = 1.0 / n
            else:
                restart[s, q] = 1.0
        x, out = restart.clone(), [None] * len(part)
        for _ in range(10000):
            y = torch.zeros_like(x).index_add_(0, dst, (x * inv[:, None])[src])
            y = (1.0 - DAMPING) * restart + DAMPING * y
            change = (y - x).abs().sum(0).tolist()
            x = y
            for q, r in enumerate(change):
                if out[q] is None and r < EPSILON:
                    out[q] = x[:, q].cpu().numpy()
            if all(o is not None for o in out):
                break
        cols += out
    return cols


def _hub(n, src):
    deg = torch.bincount(src.long(), minlength=n)
    return int((deg == deg.max()).nonzero()[0])


def exact(case, seed):
    """PageRank in 64 bits; the labels of the other algorithms are whole numbers."""
    if case["kind"] == "packed":
        return None
    if case["kind"] == "serve":
        n, src, dst, _ = _edges(case, seed)
        stream = _stream(case, seed, n, _hub(n, src))
        ranks = iter(_pagerank64(n, src, dst, [s for a, s in stream if a == "ppr"]))
        return [next(ranks) if a == "ppr" else None for a, _ in stream]
    if case["algo"] not in ("pr", "ppr"):
        return None
    n, src, dst, _ = _edges(case, seed)
    if case["kind"] == "batch":
        return np.stack(_pagerank64(n, src, dst, [int(s) for s in _sources(case, seed, n)]))
    return _pagerank64(n, src, dst, [None if case["algo"] == "pr" else _hub(n, src)])[0]
