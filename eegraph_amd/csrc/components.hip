// Connected components by union-find, for the variants of CC that only ask for the labels.
//
// The reference propagates minimum labels along every edge until nothing changes (src/cc.cu:
// 26-271); relax.hip does the same over the symmetrised list: two sweeps over 2m edges on
// RMAT-22, each bound by a 4-byte gather per edge.  Most of those edges join vertices that two
// edges per vertex have already joined.  As in Afforest (Sutton, Ben-Nun, Barak, "Optimizing
// Parallel Graph Connectivity Computation via Subgraph Sampling", IPDPS 2018), the first edges of
// every vertex are linked, the most frequent component of a sample is taken for the giant one, and
// only edges that leave other vertices are looked at afterwards.  With the symmetrised list at
// hand, vertices of the giant component are skipped altogether (every edge to them is seen from
// its other end); without it (it costs a sort of 2m edges) the edges are read once and those
// inside the giant component are dropped by a bit per endpoint.
//
// parent[] holds internal ids that only decrease along a path, so there are no cycles.  In the last
// links a root is only ever changed by a compare-and-swap, so a stale read shows an earlier ancestor
// and costs a step, never a lost link, and shortcuts are stored past the caches (agent scope).  The label of a
// component is its smallest original id, as everywhere: whatever the order of the links, the
// answer is unique.
// Measured, device time against label propagation: RMAT-22 1.89 -> 0.20 ms with the symmetrised
// list and 0.64 without (which saves its sort of 134 M pairs), 4096^2 grid 33 -> 1.6 / 1.8 ms,
// RMAT-14 0.20 -> 0.04 / 0.05 ms.  Bound by the line fetched for the first edges of every vertex.
#include <algorithm>
#include <chrono>

#include "engine.hpp"

namespace eeg {
namespace {

constexpr int CC_NBRS = 2;          // edges of every vertex linked before the sample
constexpr int CC_UNIT = WAVE;       // edges of a non-giant vertex that a wave takes at once
constexpr int CC_CHUNK = 8 * WG;    // edges per workgroup without the symmetrised list
constexpr int CC_SAMPLE = 256;

unsigned cc_grid(uint64_t work, unsigned cap = 8192) {
    return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(cap, (work + WG - 1) / WG));
}

__device__ __forceinline__ uint32_t cc_root(uint32_t* parent, uint32_t x) {
    uint32_t p = parent[x];
    while (p != x) {
        const uint32_t g = parent[p];
        if (g != p) __hip_atomic_store(&parent[x], g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        x = p;
        p = g;
    }
    return x;
}

// Joins the components of u and v.  Every lane of the wave calls it (on: the lane has an edge):
// neighbouring lanes often hold the same pair of roots, which is linked once, and a root is read
// past the caches before the compare-and-swap, since a cached copy keeps showing a root to all its
// vertices after it has been linked (4096^2 grid: the first links 4.5-7.2 ms without both, 1.5-1.7 ms with).
__device__ __forceinline__ void cc_link(uint32_t* parent, uint32_t u, uint32_t v, bool on) {
    uint32_t a = on ? cc_root(parent, u) : 0u, b = on ? cc_root(parent, v) : 0u;
    const uint32_t pa = __shfl_up(a, 1, WAVE), pb = __shfl_up(b, 1, WAVE);
    if (lane_id() && min(a, b) == min(pa, pb) && max(a, b) == max(pa, pb)) return;
    while (a != b) {
        const uint32_t hi = max(a, b), lo = min(a, b);
        uint32_t p = __hip_atomic_load(&parent[hi], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (p == hi) {
            p = atomicCAS(&parent[hi], hi, lo);
            if (p == hi) return;
        }
        // hi had a parent already: go on from there
        a = cc_root(parent, p);
        b = lo;
        if (a != b) b = cc_root(parent, b);
    }
}

// Every vertex below its first neighbour's id, or its own root; smallest original id seen so far.
__global__ void k_cc_init(const uint64_t* __restrict__ row, const uint32_t* __restrict__ col, uint32_t n,
                          const uint32_t* __restrict__ inv, uint32_t* __restrict__ parent,
                          uint32_t* __restrict__ minid, Ctl* ctl) {
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl->qpack[0] = 0;
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
         v += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t r0 = row[v];
        uint32_t p = (uint32_t)v;
        if (row[v + 1] > r0) p = min(p, col[r0]);
        parent[v] = p;
        minid[v] = inv[v];
    }
}

// Root of v, which v points at afterwards (no links run beside it, so roots stay roots).  Mostly a step
// or two away.  Where first edges form a long chain (a wheel whose rim is listed first: a vertex a step,
// although all vertices have a neighbour in common) the lanes on it jump: each stores how far it has got
// and reads on from there past the caches, so that the distance doubles with every step of the lanes
// that are under way.  The lanes above them come later, so a thread takes one vertex and the grid is as
// large as the graph.  Device time on wheels of 2^20 / 2^22 vertices, walking only, with a grid of 8192
// workgroups: 3.8 / 162 ms; now 0.27 / 0.75 (label propagation 0.19 / 0.68).  Walks up to CC_STEPS are
// cheaper in the caches: jumping after 64 steps costs the 2048^2 grid 0.61 ms, after 128 0.55 as without.
constexpr int CC_STEPS = 128;
__device__ __forceinline__ uint32_t cc_settle(uint32_t* parent, uint32_t v) {
    const uint32_t p = parent[v];
    uint32_t r = p, g = parent[r];
    for (int k = 0; k < CC_STEPS && g != r; ++k) {
        r = g;
        g = parent[r];
    }
    while (g != r) {
        r = g;
        __hip_atomic_store(&parent[v], r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        g = __hip_atomic_load(&parent[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (r != p) parent[v] = r;
    return r;
}

// Every vertex points at its root.
__global__ void k_cc_compress(uint32_t* parent, uint32_t n) {
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
         v += (uint64_t)gridDim.x * blockDim.x)
        (void)cc_settle(parent, (uint32_t)v);
}

// First edges: the larger of two roots below the smaller.  Plain stores: of two links of the same
// root one is lost, which only leaves a smaller giant component (compare-and-swaps queued on the
// hubs' roots: 1270 us on RMAT-22, as stores 70).  Roots are one step away here.
__global__ void k_cc_hook_first(const uint64_t* __restrict__ row, const uint32_t* __restrict__ col, uint32_t n,
                                uint32_t* parent) {
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
         v += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t r0 = row[v], r1 = row[v + 1];
        for (int k = 0; k < CC_NBRS && r0 + k < r1; ++k) {
            const uint32_t a = parent[v], b = parent[col[r0 + k]];
            if (a != b) parent[max(a, b)] = min(a, b);
        }
    }
}

// The same edges again, none lost, for the vertices outside the giant component so far: few
// where there are hubs, most of a grid (whose hooks only merge neighbours).
__global__ void k_cc_link_first(const uint64_t* __restrict__ row, const uint32_t* __restrict__ col, uint32_t n,
                                uint32_t* parent, const uint32_t* __restrict__ giant) {
    const uint32_t gr = *giant;
    for (uint64_t b = (uint64_t)blockIdx.x * blockDim.x; b < n; b += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t v = b + threadIdx.x;
        const bool on = v < n && parent[v] != gr;
        if (!__ballot(on)) continue;
        const uint64_t r0 = on ? row[v] : 0, r1 = on ? row[v + 1] : 0;
        for (int k = 0; k < CC_NBRS; ++k) {
            const bool edge = r0 + k < r1;
            cc_link(parent, (uint32_t)v, edge ? col[r0 + k] : 0u, edge);
        }
    }
}

// The most frequent root among the ends of CC_SAMPLE edges spread over the list (one workgroup).
__global__ __launch_bounds__(CC_SAMPLE) void k_cc_sample(const uint32_t* __restrict__ col, uint64_t m,
                                                         const uint32_t* __restrict__ parent, uint32_t* giant) {
    __shared__ uint32_t s[CC_SAMPLE];
    __shared__ unsigned long long best;
    const uint32_t i = threadIdx.x;
    const uint32_t r = parent[col[m / CC_SAMPLE * i + m % CC_SAMPLE * i / CC_SAMPLE]];
    s[i] = r;
    if (i == 0) best = 0;
    __syncthreads();
    uint32_t cnt = 0;
    for (int k = 0; k < CC_SAMPLE; ++k) cnt += s[k] == r;
    atomicMax(&best, ((unsigned long long)cnt << 32) | r);
    __syncthreads();
    if (i == 0) *giant = (uint32_t)best;
}

// Vertices outside the giant component with more than the first edges, which k_cc_link_first has linked
// (it left out only vertices of that component): queue q, prefix s of their units of CC_UNIT edges,
// totals in ctl->qpack[0].  A wave takes a unit, so vertices of one or two edges would leave it all but
// idle (1000 stars of 1000 vertices: 0.34 ms with them, 0.05 without; label propagation 0.18).
__global__ __launch_bounds__(WG) void k_cc_collect(const uint64_t* __restrict__ row, uint32_t n,
                                                   const uint32_t* __restrict__ parent,
                                                   const uint32_t* __restrict__ giant, uint32_t* __restrict__ q,
                                                   uint32_t* __restrict__ s, Ctl* ctl) {
    __shared__ uint64_t sScan[WG / WAVE + 1];
    __shared__ unsigned long long sBase;
    const uint32_t gr = parent[*giant];
    for (uint64_t b = (uint64_t)blockIdx.x * WG; b < n; b += (uint64_t)gridDim.x * WG) {
        const uint64_t v = b + threadIdx.x;
        uint64_t mine = 0;
        if (v < n && parent[v] != gr) {
            const uint64_t d = row[v + 1] - row[v];
            if (d > CC_NBRS) mine = 1ull | ((d - CC_NBRS + CC_UNIT - 1) / CC_UNIT << 32);
        }
        if (!__syncthreads_or(mine != 0)) continue;  // the same answer in every thread
        uint64_t tot;
        const uint64_t pre = block_excl_scan<uint64_t>(mine, sScan, &tot);
        if (threadIdx.x == 0) sBase = atomicAdd(&ctl->qpack[0], (unsigned long long)tot);
        __syncthreads();
        if (mine) {
            const uint32_t pos = (uint32_t)sBase + (uint32_t)pre;
            q[pos] = (uint32_t)v;  // pos < n: a vertex is queued once
            s[pos] = (uint32_t)(sBase >> 32) + (uint32_t)(pre >> 32);
        }
        __syncthreads();
    }
}

// Links the edges of the queued vertices beyond the first: a wave per unit, a contiguous run of units per wave.
__global__ __launch_bounds__(WG) void k_cc_link_queue(const uint64_t* __restrict__ row, const uint32_t* __restrict__ col,
                                                      const uint32_t* __restrict__ q, const uint32_t* __restrict__ s,
                                                      const Ctl* ctl, uint32_t* parent) {
    const unsigned long long pk = ctl->qpack[0];
    const uint32_t nE = (uint32_t)pk, T = (uint32_t)(pk >> 32);
    const uint32_t lane = (uint32_t)lane_id();
    const uint64_t nw = (uint64_t)gridDim.x * (WG / WAVE);
    const uint64_t w = (uint64_t)blockIdx.x * (WG / WAVE) + threadIdx.x / WAVE;
    const uint32_t t0 = (uint32_t)(w * T / nw), t1 = (uint32_t)((w + 1) * T / nw);
    if (t0 >= t1) return;
    uint32_t lo = 0, hi = nE;  // last entry with s <= t0: 64 positions a step
    while (hi - lo > 1) {
        const uint32_t step = (hi - lo + WAVE - 1) / WAVE;
        const uint64_t i = (uint64_t)lo + (uint64_t)lane * step;
        const uint64_t below = __ballot(i < hi && s[i] <= t0);  // lane 0 always: s[lo] <= t0
        lo += (uint32_t)(__popcll((unsigned long long)below) - 1) * step;
        hi = min(hi, lo + step);
    }
    for (uint32_t t = t0; t < t1; ++t) {
        while (lo + 1 < nE && s[lo + 1] <= t) ++lo;
        const uint32_t v = q[lo];
        const uint64_t e = row[v] + CC_NBRS + (uint64_t)(t - s[lo]) * CC_UNIT + lane;
        const bool edge = e < row[v + 1];
        cc_link(parent, v, edge ? col[e] : 0u, edge);
    }
}

// bit v % 64 of word v / 64: v is in the giant component
__global__ void k_cc_giant_bits(const uint32_t* __restrict__ parent, uint32_t n, const uint32_t* __restrict__ giant,
                                uint64_t* __restrict__ bits) {
    const uint32_t gr = parent[*giant];
    const uint64_t nw = ((uint64_t)n + 63) / 64;
    for (uint64_t w = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / WAVE; w < nw;
         w += (uint64_t)gridDim.x * blockDim.x / WAVE) {
        const uint64_t v = w * 64 + (uint64_t)lane_id();
        const uint64_t b = __ballot(v < n && parent[v] == gr);
        if (lane_id() == 0) bits[w] = b;
    }
}

// Every edge that is not inside the giant component, linked; 8 consecutive edges per thread.
__global__ __launch_bounds__(WG) void k_cc_link_edges(const uint64_t* __restrict__ row, const uint32_t* __restrict__ col,
                                                      uint32_t n, uint64_t m, const uint32_t* __restrict__ bits,
                                                      uint32_t* parent) {
    __shared__ uint32_t sEnd;
    auto in = [&](uint32_t v) { return (bits[v >> 5] >> (v & 31u)) & 1u; };
    const uint64_t chunks = (m + CC_CHUNK - 1) / CC_CHUNK;
    for (uint64_t c = blockIdx.x; c < chunks; c += gridDim.x) {
        const uint64_t e0 = c * CC_CHUNK, e1 = min(e0 + (uint64_t)CC_CHUNK, m);
        // sources of the chunk's first and last edge: threads 0 and 1 search, then every thread
        // searches between them
        __syncthreads();
        __shared__ uint32_t sBeg;
        if (threadIdx.x < 2) {
            const uint64_t e = threadIdx.x ? e1 - 1 : e0;
            uint32_t lo = 0, hi = n;  // last v with row[v] <= e
            while (hi - lo > 1) {
                const uint32_t mid = lo + (hi - lo) / 2;
                if (row[mid] <= e) lo = mid; else hi = mid;
            }
            if (threadIdx.x) sEnd = lo;
            else sBeg = lo;
        }
        __syncthreads();
        uint64_t e = e0 + 8ull * threadIdx.x;
        const bool any = e < e1;
        uint32_t u[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) u[k] = e + k < e1 ? col[e + k] : 0u;
        uint32_t lo = sBeg, hi = any ? sEnd + 1 : lo + 1;
        while (hi - lo > 1) {
            const uint32_t mid = lo + (hi - lo) / 2;
            if (row[mid] <= e) lo = mid; else hi = mid;
        }
        uint64_t end = row[lo + 1];
        bool mine = in(lo);
#pragma unroll
        for (int k = 0; k < 8; ++k, ++e) {
            const bool edge = e < e1;
            while (edge && e >= end) {
                end = row[++lo + 1];
                mine = in(lo);
            }
            const bool link = edge && !(mine && in(u[k]));
            if (__ballot(link)) cc_link(parent, lo, u[k], link);
        }
    }
}

// Roots for good, and the smallest original id of each: non-roots offer theirs to their root, one
// atomic per wave for the root of its first lane, none where the id at hand (it only falls) is
// already smaller.
__global__ void k_cc_min(uint32_t* parent, uint32_t n, const uint32_t* __restrict__ inv, uint32_t* minid) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t b = (uint64_t)blockIdx.x * blockDim.x; b < n; b += stride) {
        const uint64_t v = b + threadIdx.x;
        uint32_t r = 0xffffffffu, id = 0xffffffffu;
        if (v < n) {
            r = cc_settle(parent, (uint32_t)v);
            if (r != v) id = inv[v];
        }
        const uint32_t r0 = __builtin_amdgcn_readfirstlane(r);
        uint32_t best = r == r0 ? id : 0xffffffffu;
#pragma unroll
        for (int off = WAVE / 2; off > 0; off >>= 1) best = min(best, (uint32_t)__shfl_xor(best, off, WAVE));
        const bool offer = r == r0 ? lane_id() == 0 : id != 0xffffffffu;
        if (r == r0) id = best;
        if (offer && id != 0xffffffffu && id < minid[r]) atomicMin(&minid[r], id);
    }
}

__global__ void k_cc_label(const uint32_t* __restrict__ parent, uint32_t n, const uint32_t* __restrict__ minid,
                           uint32_t* __restrict__ lab) {
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
         v += (uint64_t)gridDim.x * blockDim.x)
        lab[v] = minid[parent[v]];
}

}  // namespace

eeg_status run_components(eeg_graph* g, eeg_stats* st, Work& w, hipStream_t s) {
    const auto t_host0 = std::chrono::steady_clock::now();
    const uint32_t n = g->n;
    // (the limit of the symmetrised list holds with and without it)
    if (2 * g->m >= 0xffffffffull)
        return fail(EEG_ERR_UNSUPPORTED, "symmetrised edge count exceeds 2^32-1");
    const bool sym = g->sym.built;
    const Csr& c = sym ? g->sym : g->out;
    for (DevMem* d : {&w.lab, &w.q[0], &w.s[0], &w.q[1], &w.s[1]}) EEG_TRY(d->alloc((size_t)n * 4 + 8));
    EEG_TRY(w.ctl.alloc(sizeof(Ctl)));
    uint32_t* parent = w.q[0].as<uint32_t>();
    uint32_t* minid = w.s[0].as<uint32_t>();
    Ctl* ctl = w.ctl.as<Ctl>();
    uint32_t* giant = &ctl->iters;
    const uint32_t* inv = g->inv.as<uint32_t>();
    hipEvent_t e0, e1;
    EEG_TRY(w.event(0, &e0));
    EEG_TRY(w.event(1, &e1));
    EEG_HIP(hipEventRecord(e0, s));
    const unsigned gn = cc_grid(n), gv = cc_grid(n, 0xffffffu);  // (a launch holds fewer than 2^32 threads)
    uint32_t launches = 3;
    k_cc_init<<<gn, WG, 0, s>>>(c.rowp(), c.colp(), n, inv, parent, minid, ctl);
    if (c.m) {
        k_cc_compress<<<gv, WG, 0, s>>>(parent, n);
        k_cc_hook_first<<<gn, WG, 0, s>>>(c.rowp(), c.colp(), n, parent);
        k_cc_compress<<<gv, WG, 0, s>>>(parent, n);
        k_cc_sample<<<1, CC_SAMPLE, 0, s>>>(c.colp(), c.m, parent, giant);
        k_cc_link_first<<<gn, WG, 0, s>>>(c.rowp(), c.colp(), n, parent, giant);
        k_cc_compress<<<gv, WG, 0, s>>>(parent, n);
        if (sym) {
            k_cc_collect<<<gn, WG, 0, s>>>(c.rowp(), n, parent, giant, w.q[1].as<uint32_t>(), w.s[1].as<uint32_t>(), ctl);
            k_cc_link_queue<<<2048, WG, 0, s>>>(c.rowp(), c.colp(), w.q[1].as<uint32_t>(), w.s[1].as<uint32_t>(), ctl, parent);
        } else {
            k_cc_giant_bits<<<gn, WG, 0, s>>>(parent, n, giant, w.q[1].as<uint64_t>());
            k_cc_link_edges<<<(unsigned)std::min<uint64_t>(8192, (c.m + CC_CHUNK - 1) / CC_CHUNK), WG, 0, s>>>(
                c.rowp(), c.colp(), n, c.m, w.q[1].as<uint32_t>(), parent);
        }
        launches += 8;
    }
    k_cc_min<<<gv, WG, 0, s>>>(parent, n, inv, minid);
    k_cc_label<<<gn, WG, 0, s>>>(parent, n, minid, w.lab.as<uint32_t>());
    EEG_HIP(hipGetLastError());
    EEG_HIP(hipEventRecord(e1, s));
    EEG_HIP(hipStreamSynchronize(s));
    if (st) {
        float ms = 0;
        EEG_HIP(hipEventElapsedTime(&ms, e0, e1));
        st->iterations = c.m ? 2 : 1;  // the sampled links and the remaining ones
        st->launches = launches;
        st->ms_traversal = ms;
        st->ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_host0).count();
    }
    return EEG_OK;
}

}  // namespace eeg
