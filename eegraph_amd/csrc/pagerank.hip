// PageRank and personalised PageRank.
//
// The reference pushes float deltas with atomicAdd (src/pr.cu:3-288): the order of additions
// changes from run to run and every part of a multi-part vertex consumes the same delta
// (D6).  Here:
//   sync variants  - Jacobi iteration x' = (1-d)/N + d * sum_{u->v} x_u/outdeg(u), x0 = 1/N,
//                    gathered per destination over the in-edge list (k_pr_stream, then
//                    k_pr_finish): 16 consecutive in-edges per lane summed with compensation
//                    (TwoSum), rows that cross lanes joined by a segmented scan, rows that cross
//                    wave tiles by their tiles' tails in tile order.  The order of every sum is
//                    fixed, so results are deterministic.
//                    The L1 residual is accumulated in FP64 and reduced in a fixed order.
//   async variants - a gather with ranks updated in place (Gauss-Seidel in tile order,
//                    k_pr_pull): Tigr virtual nodes of K in-edges, K lanes and one edge per
//                    lane, a TwoSum tree per virtual node, each vertex's virtual nodes of a tile
//                    in order, vertices that span tiles finished by a fix-up pass in tile order.
//                    Fewer sweeps, no atomics, order of reads not fixed (result within the
//                    tolerance, not bit-reproducible).  The sync variants run this kernel too
//                    (out of place, deterministic) where the stream tables do not fit in memory.
//   personalised   - the same iterations with a one-hot restart: x0 = e_s and
//                    x' = (1-d) e_s + d * sum_{u->v} x_u/outdeg(u), stopped at the same L1
//                    residual.  A residual push with a per-vertex threshold small enough for
//                    an L1 bound of 1e-7 at N = 2^26 touches every vertex many times with float
//                    atomics; the gather does each iteration in one pass without atomics.
//   Mass of vertices without out-edges is dropped (not redistributed) in both forms.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <vector>

#include "compensated.hpp"
#include "engine.hpp"

namespace eeg {
namespace {

struct PullArgs {
    const uint64_t* row;     // in-edge CSR
    const uint32_t* col;     // sources of in-edges
    const uint32_t* vlist;   // vertices with in-edges
    const uint32_t* vscan;   // their virtual-node prefix
    uint32_t nz;
    uint32_t P;
    const float* c_old;      // contributions x_u / outdeg(u)
    const float* x_old;      // ranks as compensated pairs: x = hi + lo
    const float* xl_old;
    float* x_new;
    float* xl_new;
    float* c_new;
    const uint32_t* outdeg;  // out-degrees for the new contributions
    float2* spill;           // per tile: head and tail partials
    double* res_part;        // per workgroup FP64 residual
    Ctl* ctl;
    float base;              // teleport term of every vertex: (1-d)/N, or 0 when personalised
    float damping;
    uint32_t it;
    uint32_t pers;           // personalised: restart vertex (internal id), else 0xffffffff
    float pers_base;         // its teleport term, 1-d
    uint32_t strided;        // in place: workgroup b takes tiles b, b + grid, ... (see k_pr_pull)
    const uint32_t* tstart;  // first entry of each tile (vlist position)
    float* cerr;             // per vertex: rounding error of its last contribution (null: dropped)
};

// New rank of v from its gathered sum; xo = old rank (hi + lo), d = out-degree.
__device__ __forceinline__ void finish_vertex(const PullArgs& a, uint32_t v, Comp sum, double xo, uint32_t d,
                                              uint32_t feed, double& res) {
    float hi, lo;
    rank_pair(v == a.pers ? a.pers_base : a.base, a.damping, sum, &hi, &lo);
    a.x_new[v] = hi;
    a.xl_new[v] = lo;
    float c = contribution(hi, lo, d);
    if (feed & FEED_WRITE) {
        float e = (feed & FEED_READ) ? a.cerr[v] : 0.0f;
        c = fed_contribution(c, hi, lo, d, &e);
        a.cerr[v] = e;
    }
    a.c_new[v] = c;
    res += fabs(((double)hi + (double)lo) - xo);
}

// Edge slots per pull tile: twice the traversal tile, so each lane keeps 16 independent
// gathers in flight and the per-tile staging is amortised over more edges.
constexpr int PR_TILE = 2 * TILE_EDGES;
// Virtual nodes of one entry in one tile beyond which a wave, not a thread, sums them.
constexpr int PR_LONG = 32;

// FEED: rounding errors are fed back where the control block says so (a kernel of its own, which runs once
// the host has seen that: 14.2 us a sweep of RMAT-16 against 13.2).
template <int K, bool FEED>
// At most 64 VGPRs, 8 waves per SIMD (K = 4: LDS holds 4 workgroups per CU, so 128): the
// gathers are latency-bound, so the extra resident waves are worth more than the registers
// (-4% per iteration against 71 VGPRs, 7 waves, at K = 8).
__global__ __launch_bounds__(WG, K >= 8 ? 8 : 4) void k_pr_pull(PullArgs a) {
    constexpr int VPR = WG / K;
    constexpr int TV = PR_TILE / K;
    constexpr int ROUNDS = PR_TILE / WG;
    constexpr int EMAX = TV + 2;
    __shared__ uint32_t sS[EMAX];
    __shared__ uint64_t sRow[EMAX];
    __shared__ uint32_t sDeg[EMAX];
    __shared__ uint16_t sOwn[TV];
    __shared__ float2 sPart[TV];
    __shared__ float2 sXo[EMAX];     // old rank (hi, lo) of each entry, loaded with its row
    __shared__ uint32_t sOd[EMAX];   // out-degree of each entry
    __shared__ double sRed[WG / WAVE];

    if (a.ctl->done) return;
    const uint32_t feed = FEED ? a.ctl->feed : 0u;
    double res = 0.0;
    const uint32_t T = a.P, nE = a.nz;
    const uint32_t ntiles = (T + TV - 1) / TV;
    const uint32_t c0 = (uint32_t)((uint64_t)blockIdx.x * ntiles / gridDim.x);
    const uint32_t c1 = (uint32_t)((uint64_t)(blockIdx.x + 1) * ntiles / gridDim.x);
    const int grp = threadIdx.x / K, lj = threadIdx.x % K;
    // Tiles: a contiguous run per workgroup, or (in place) strided over the grid, so the first
    // tiles of every workgroup - the highest-degree vertices in degree order, whose
    // contributions most edges gather - are finished in the first round and the later rounds
    // already read their new values (Gauss-Seidel by rounds of `grid` tiles).
    const uint32_t tb = a.strided ? blockIdx.x : c0, te = a.strided ? ntiles : c1;
    const uint32_t tstep = a.strided ? gridDim.x : 1u;
    if (tb < te) {
        uint32_t e_start = a.tstart[tb];
        for (uint32_t tile = tb; tile < te; tile += tstep) {
            const uint32_t t0 = tile * TV;
            const uint32_t t1 = min(t0 + (uint32_t)TV, T);
            // the entry holding vnode t1 (the next tile's first entry; nE past the last tile):
            // at most TV entries start in (t0, t1], so it lies within the staged window
            const uint32_t e_next = (tile + 1 < ntiles) ? a.tstart[tile + 1] : nE;
            for (int k = threadIdx.x; k < EMAX; k += WG) {
                const uint64_t i = (uint64_t)e_start + k;
                sS[k] = (i <= nE) ? a.vscan[i] : 0xffffffffu;  // vscan[nE] = P closes the last
            }
            __syncthreads();
            // entries in the tile: up to e_next, and e_next itself when it starts before t1
            const int nent = (int)(e_next - e_start) + (sS[e_next - e_start] < t1 ? 1 : 0);
            // entry data, including what finishing the vertex needs, so those loads overlap
            // with the row loads instead of trailing the gathers
            for (int k = threadIdx.x; k < nent; k += WG) {
                const uint32_t v = a.vlist[e_start + k];
                const uint64_t r0 = a.row[v];
                sRow[k] = r0;
                sDeg[k] = (uint32_t)(a.row[v + 1] - r0);
                sXo[k] = make_float2(a.x_old[v], a.xl_old[v]);
                sOd[k] = a.outdeg[v];
            }
            for (int j = threadIdx.x; j < (int)(t1 - t0); j += WG) {
                const uint32_t t = t0 + j;
                int lo = 0, hi = nent;
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (sS[mid] <= t) lo = mid; else hi = mid;
                }
                sOwn[j] = (uint16_t)lo;
            }
            __syncthreads();
            // one in-edge per lane, K lanes per virtual node, TwoSum tree per virtual node;
            // the source indices of all rounds are loaded first, then all contributions, so a
            // lane keeps ROUNDS independent requests in flight
            // Branch-free rounds: a slot past the tile or past its virtual node's edges reads
            // edge 0 and its contribution (always in range, and one shared address per wave)
            // and drops the value, so no exec-mask branches surround the loads.
            uint32_t pidx[ROUNDS];
            bool pv[ROUNDS];
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r) {
                const int slot = r * VPR + grp;  // < TV: sOwn[slot] is in range
                const uint32_t t = t0 + slot;
                const bool tin = t < t1;
                const int k = tin ? (int)sOwn[slot] : 0;
                const uint32_t eoff = (t - sS[k]) * K + lj;
                pv[r] = tin && eoff < sDeg[k];
                const uint64_t e = pv[r] ? sRow[k] + eoff : 0ull;
                // streamed once per iteration: keep it from evicting the gathered contributions
                pidx[r] = __builtin_nontemporal_load(&a.col[e]);
            }
            float pc[ROUNDS];
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r) {
                const float c = a.c_old[pidx[r]];
                pc[r] = pv[r] ? c : 0.0f;
            }
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r) {
                const int slot = r * VPR + grp;
                const Comp g = group_sum_first_lane<K>(pc[r]);
                if (lj == 0 && t0 + slot < t1) sPart[slot] = make_float2(g.s, g.e);
            }
            __syncthreads();
            // Per entry: its virtual nodes of this tile added in order, one thread per entry.  A
            // run longer than PR_LONG (the hubs: up to a whole tile) is summed by one wave
            // instead, each lane a contiguous chunk in order and the lanes by a fixed tree, so a
            // single thread does not serialise the tile.
            auto finish_entry = [&](int k, Comp acc) {
                const bool started_before = sS[k] < t0;
                const bool continues = sS[k + 1] > t1;
                if (!started_before && !continues) {
                    const float2 xo = sXo[k];
                    finish_vertex(a, a.vlist[e_start + k], acc, (double)xo.x + (double)xo.y, sOd[k], feed, res);
                } else if (started_before) {
                    a.spill[2 * tile] = make_float2(acc.s, acc.e);      // head
                } else {
                    a.spill[2 * tile + 1] = make_float2(acc.s, acc.e);  // tail
                }
            };
            for (int k = threadIdx.x; k < nent; k += WG) {
                const uint32_t s0 = max(sS[k], t0), s1 = min(sS[k + 1], t1);
                if (s1 - s0 > (uint32_t)PR_LONG) continue;
                Comp acc{0.0f, 0.0f};
                for (uint32_t t = s0; t < s1; ++t) {
                    const float2 p = sPart[t - t0];
                    acc = comp_add(acc, Comp{p.x, p.y});
                }
                finish_entry(k, acc);
            }
            {
                const int wv = threadIdx.x / WAVE, lane = (int)lane_id();
                int nlong = 0;  // long entries seen so far; the j-th goes to wave j % waves
                for (int base = 0; base < nent; base += WAVE) {
                    const int k = base + lane;
                    bool lng = false;
                    if (k < nent) lng = min(sS[k + 1], t1) - max(sS[k], t0) > (uint32_t)PR_LONG;
                    uint64_t mask = __ballot(lng);
                    while (mask) {
                        const int kk = base + (int)(__ffsll((unsigned long long)mask) - 1);
                        mask &= mask - 1;
                        if (nlong++ % (WG / WAVE) != wv) continue;
                        const uint32_t s0 = max(sS[kk], t0), s1 = min(sS[kk + 1], t1);
                        const uint32_t chunk = (s1 - s0 + WAVE - 1) / WAVE;
                        const uint32_t q0 = min(s0 + (uint32_t)lane * chunk, s1), q1 = min(q0 + chunk, s1);
                        Comp acc{0.0f, 0.0f};
                        for (uint32_t t = q0; t < q1; ++t) {
                            const float2 p = sPart[t - t0];
                            acc = comp_add(acc, Comp{p.x, p.y});
                        }
#pragma unroll
                        for (int off = WAVE / 2; off > 0; off >>= 1) {
                            Comp o;
                            o.s = __shfl_down(acc.s, off, WAVE);
                            o.e = __shfl_down(acc.e, off, WAVE);
                            acc = comp_add(acc, o);
                        }
                        if (lane == 0) finish_entry(kk, acc);
                    }
                }
            }
            __syncthreads();
            if (!a.strided) e_start = e_next;
            else if (tile + tstep < te) e_start = a.tstart[tile + tstep];
        }
    }
    // fixed-order block reduction of the FP64 residual
    res = wave_sum(res);
    if (lane_id() == 0) sRed[threadIdx.x / WAVE] = res;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int i = 0; i < WG / WAVE; ++i) t += sRed[i];
        a.res_part[blockIdx.x] = t;
    }
}

// Tiles crossed by a vertex beyond which a wave, not a thread, combines its partial sums.
constexpr uint32_t FIX_LONG = 8;

// Vertices whose virtual nodes span tiles: tail of the first tile + heads of the following
// tiles, in tile order.  `span` lists their vlist positions: one thread per vertex, and one
// wave per vertex in `span_long` (the hubs, crossing more than FIX_LONG tiles), whose lanes
// load the partial sums at once and whose lane 0 adds them in the same order.
__global__ __launch_bounds__(WG) void k_pr_fix(PullArgs a, const uint32_t* __restrict__ span, uint32_t nspan,
                                               const uint32_t* __restrict__ span_long, uint32_t nlong,
                                               uint32_t TV, double* res_part) {
    __shared__ double sRed[WG / WAVE];
    if (a.ctl->done) return;
    const uint32_t feed = a.cerr ? a.ctl->feed : 0u;
    double res = 0.0;
    for (uint32_t i = blockIdx.x * WG + threadIdx.x; i < nspan; i += gridDim.x * WG) {
        const uint32_t pos = span[i];
        const uint32_t s0 = a.vscan[pos], s1 = a.vscan[pos + 1];
        const uint32_t ta = s0 / TV, tb = (s1 - 1) / TV;
        const float2 tl = a.spill[2 * ta + 1];
        Comp acc{tl.x, tl.y};
        for (uint32_t t = ta + 1; t <= tb; ++t) {
            const float2 h = a.spill[2 * t];
            acc = comp_add(acc, Comp{h.x, h.y});
        }
        const uint32_t v = a.vlist[pos];
        finish_vertex(a, v, acc, (double)a.x_old[v] + (double)a.xl_old[v], a.outdeg[v], feed, res);
    }
    const int lane = (int)lane_id();
    const uint32_t nw = gridDim.x * (WG / WAVE);
    for (uint32_t j = blockIdx.x * (WG / WAVE) + threadIdx.x / WAVE; j < nlong; j += nw) {
        const uint32_t pos = span_long[j];
        const uint32_t s0 = a.vscan[pos], s1 = a.vscan[pos + 1];
        const uint32_t ta = s0 / TV, np = (s1 - 1) / TV - ta + 1;  // parts: tail of ta, heads after
        // starting from 0 + tail gives the tail's bits exactly, as the thread form does
        Comp acc{0.0f, 0.0f};
        for (uint32_t base = 0; base < np; base += WAVE) {
            const uint32_t p = base + (uint32_t)lane;
            float2 h = make_float2(0.0f, 0.0f);
            if (p < np) h = a.spill[p == 0 ? 2 * ta + 1 : 2 * (ta + p)];
            const uint32_t cnt = min(np - base, (uint32_t)WAVE);
            for (uint32_t l = 0; l < cnt; ++l) {
                const float hs = __shfl(h.x, (int)l, WAVE), he = __shfl(h.y, (int)l, WAVE);
                acc = comp_add(acc, Comp{hs, he});
            }
        }
        if (lane == 0) {
            const uint32_t v = a.vlist[pos];
            finish_vertex(a, v, acc, (double)a.x_old[v] + (double)a.xl_old[v], a.outdeg[v], feed, res);
        }
    }
    res = wave_sum(res);
    if (lane_id() == 0) sRed[threadIdx.x / WAVE] = res;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int i = 0; i < WG / WAVE; ++i) t += sRed[i];
        res_part[blockIdx.x] = t;
    }
}

// Vertices without in-edges hold their teleport term from the first iteration on.  In place the old
// and the new ranks are the same memory, so the old one is read first and the pointers may alias.
__global__ void k_pr_isolated(const uint64_t* __restrict__ in_row, const uint32_t* __restrict__ outdeg,
                              uint32_t n, const float* x_old, const float* xl_old, float* x_new, float* xl_new,
                              float* __restrict__ c_new, float base0, uint32_t pers, float pers_base,
                              double* res_part, const Ctl* ctl) {
    __shared__ double sRed[WG / WAVE];
    if (ctl->done) return;
    double res = 0;
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
         v += (uint64_t)gridDim.x * blockDim.x) {
        if (in_row[v + 1] != in_row[v]) continue;
        const float base = (v == pers) ? pers_base : base0;
        const double xo = (double)x_old[v] + (double)xl_old[v];
        x_new[v] = base;
        xl_new[v] = 0.0f;
        const uint32_t d = outdeg[v];
        c_new[v] = d ? base / (float)d : 0.0f;
        res += fabs((double)base - xo);
    }
    res = wave_sum(res);
    if (lane_id() == 0) sRed[threadIdx.x / WAVE] = res;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int i = 0; i < WG / WAVE; ++i) t += sRed[i];
        res_part[blockIdx.x] = t;
    }
}

// Sums the per-workgroup residuals in a fixed order and decides convergence.
// One workgroup of RED_WG threads sums the partials in a fixed order (strided per thread, then
// a tree), so the residual is deterministic.
constexpr int RED_WG = 1024;
__global__ __launch_bounds__(RED_WG) void k_pr_reduce(const double* __restrict__ part, uint32_t nparts, Ctl* ctl,
                                                      uint32_t it, double eps, FeedRule rule,
                                                      int fed) {
    __shared__ double sRed[RED_WG];
    if (ctl->done) return;
    const double last = ctl->residual[(it - 1) & 3];
    const uint32_t was = ctl->feed;
    // strided per thread, four loads in flight, added in index order (the same sum as one at
    // a time)
    double t = 0;
    uint32_t i = threadIdx.x;
    for (; i + 3 * RED_WG < nparts; i += 4 * RED_WG) {
        const double p0 = part[i], p1 = part[i + RED_WG], p2 = part[i + 2 * RED_WG], p3 = part[i + 3 * RED_WG];
        t += p0;
        t += p1;
        t += p2;
        t += p3;
    }
    for (; i < nparts; i += RED_WG) t += part[i];
    sRed[threadIdx.x] = t;
    __syncthreads();
    for (int off = RED_WG / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) sRed[threadIdx.x] += sRed[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        ctl->feed = next_feed(sRed[0], last, rule, was, fed);
        ctl->residual[it & 3] = sRed[0];
        ctl->iters = it;
        if (sRed[0] < eps) ctl->done = 1;
    }
}

// x0 = 1/N everywhere, or e_s when personalised (pers = s)
template <bool PAIR>
__global__ void k_pr_init(const uint32_t* __restrict__ outdeg, uint32_t n, float x0, uint32_t pers,
                          float* __restrict__ x, float* __restrict__ xl, float* __restrict__ c) {
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
         v += (uint64_t)gridDim.x * blockDim.x) {
        const float xv = (pers == 0xffffffffu) ? x0 : (v == pers ? 1.0f : 0.0f);
        x[v] = xv;
        xl[v] = 0.0f;
        const uint32_t d = outdeg[v];
        const float cv = d ? xv / (float)d : 0.0f;
        if constexpr (PAIR) reinterpret_cast<float2*>(c)[v] = make_float2(cv, d ? (float)((double)xv / d - (double)cv) : 0.0f);
        else c[v] = cv;
    }
}

__global__ void k_pr_output(const float* __restrict__ hi, const float* __restrict__ lo, uint32_t n,
                            float* __restrict__ out) {
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
         v += (uint64_t)gridDim.x * blockDim.x)
        out[v] = hi[v] + lo[v];
}

__global__ void k_outdeg(const uint64_t* __restrict__ row, uint32_t n, uint32_t* __restrict__ deg) {
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
         v += (uint64_t)gridDim.x * blockDim.x)
        deg[v] = (uint32_t)(row[v + 1] - row[v]);
}

// First entry of every tile: the largest i < nz with vscan[i] <= tile * TV.
__global__ void k_tile_starts(const uint32_t* __restrict__ vscan, uint32_t nz, uint32_t TV, uint32_t ntiles,
                              uint32_t* __restrict__ tstart) {
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < ntiles; t += gridDim.x * blockDim.x) {
        const uint64_t first = (uint64_t)t * TV;
        uint32_t lo = 0, hi = nz;
        while (hi - lo > 1) {
            const uint32_t mid = lo + (hi - lo) / 2;
            if (vscan[mid] <= first) lo = mid; else hi = mid;
        }
        tstart[t] = lo;
    }
}

// Vertices crossing a tile boundary: those crossing at most FIX_LONG tiles from the front of
// `span`, the others from its back (cap entries: a boundary is crossed by one vertex at most).
__global__ void k_list_spanning(const uint32_t* __restrict__ vscan, uint32_t nz, uint32_t TV, uint32_t cap,
                                uint32_t* __restrict__ span, uint32_t* __restrict__ count) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nz;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t s0 = vscan[i], s1 = vscan[i + 1];
        const uint32_t ta = s0 / TV, tb = (s1 - 1) / TV;
        if (ta == tb) continue;
        if (tb - ta + 1 > FIX_LONG) span[cap - 1 - atomicAdd(&count[1], 1u)] = (uint32_t)i;
        else span[atomicAdd(&count[0], 1u)] = (uint32_t)i;
    }
}

// ---------------------------------------------------------------- streamed Jacobi gather
// The sync iteration as two kernels: k_pr_stream sums the contributions of every row of the
// in-edge list, k_pr_finish turns the sums into ranks.
//
// What bounds a gather of c[src] over the in-edges is not HBM but the lines that each 4-byte
// gather moves from the L2 to the CU (the K-lane pull: 0.82 line requests per edge).  In degree
// order the first PS_HUBS vertices are the sources of most edges (57% on RMAT-22), so every
// workgroup copies their contributions to LDS once (152 KB, one workgroup of 16 waves per CU)
// and only the other sources are gathered from the L2: with half the hubs (76 KB, 44% of the
// edges) a run was 13% slower.  Waves are independent: a wave takes tiles of 1024 edges, 16
// consecutive edges per lane from a copy of the list laid out for 16-byte coalesced loads, sums
// them in a register with a row-end bit per edge, and joins rows across lanes with one segmented
// scan, so there is no staging of rows, no search and no barrier between tiles.  Issuing the
// next tile's gathers before the current tile is summed (120 VGPRs) changed nothing: the
// remaining gathers are bound by their lines, 145 G/s, not by latency.
// Measured (PageRank to the 1e-7 stop on RMAT-22, 67 M edges, against the pull): 22.4 -> 14.2 ms,
// an iteration 332 + 7.9 (fix-up) + 4.6 (residual) -> 198 + 23 us; personalised, 9.9 M edges over
// 0.78 M vertices: 4.68 -> 2.85 ms.
constexpr int PS_EPL = 16;               // edges per lane
constexpr int PS_TILE = WAVE * PS_EPL;   // edges per wave tile
constexpr int PS_WG = 1024;              // threads per workgroup: 16 waves, one workgroup per CU
constexpr uint32_t PS_HUBS = 38912;      // contributions held in LDS
// A contribution rounded to one float holds the ranks within a few ulps of their fixed point
// (whatever stays inside its rounding interval is lost).  Where few vertices carry most of the
// mass and the paths between them have a period (bipartite graphs, grids), the phases of the
// iteration then settle at different points and the L1 change stays near 1e-7.  So:
// - up to PS_PAIRS vertices contributions are (hi, lo) pairs, all of them in LDS (112 of 150
//   random bipartite graphs of up to 10 vertices never met the 1e-7 stop with single floats, none
//   with pairs);
// - above, each contribution's rounding error is added to the vertex's next contribution while
//   the L1 change is above PS_FEED, so that what is passed on is right on average; below it the
//   errors are dropped, and the iteration settles on a fixed point for smaller stops.
constexpr uint32_t PS_PAIRS = PS_HUBS / 2;
constexpr double PS_FEED = 5e-8;
constexpr uint32_t PS_PARTS = 2048;      // most workgroups of k_pr_finish (residual partials)
// Lists above this size are read with nontemporal loads: one that fits the 256 MB Infinity Cache
// beside the ranks is still there in the next iteration (us per iteration, cached / nontemporal:
// 64 MiB 49.5 / 53.7, 128 MiB 94 / 104, 192 MiB 175.8 / 176.0, 256 MiB 227 / 219, 512 MiB 524 /
// 504).
constexpr uint64_t PS_STREAM_BYTES = 192ull << 20;

struct StreamArgs {
    const uint4* tcol;       // sources, tile by tile: [tile][4][lane] of 4 consecutive edges
    const uint32_t* desc;    // per lane of a tile: row-end bits | row ends before it << 16
    const uint32_t* tfirst;  // row (vlist position) of every tile's first edge
    uint32_t ntiles;
    uint32_t hubs;           // contributions in LDS: a multiple of 4, or every vertex (pairs)
    const float* c_old;
    float2* sums;            // per row: sum of its edges in the tile where it ends
    float2* tail;            // per tile: sum of the row left open at its end
    const double* parts;     // residual partials of the previous iteration
    uint32_t nparts;
    double eps;
    Ctl* ctl;
    uint32_t it;
};

// Residual of iteration a.it - 1 from its partials, in a fixed order (every workgroup gets the
// same bits); sRed: PS_WG / WAVE entries.  Records it and returns whether the run has converged.
__device__ __forceinline__ bool previous_converged(const StreamArgs& a, double* sRed) {
    double t = 0;
    for (uint32_t i = threadIdx.x; i < a.nparts; i += PS_WG) t += a.parts[i];
    t = wave_sum(t);
    if (lane_id() == 0) sRed[threadIdx.x / WAVE] = t;
    __syncthreads();
    double r = 0;
    for (int i = 0; i < PS_WG / WAVE; ++i) r += sRed[i];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.ctl->residual[(a.it - 1) & 3] = r;
        a.ctl->iters = a.it - 1;
        if (r < a.eps) a.ctl->done = 1;
    }
    return r < a.eps;
}

__global__ __launch_bounds__(PS_WG) void k_pr_check(StreamArgs a) {
    __shared__ double sRed[PS_WG / WAVE];
    if (a.ctl->done) return;
    (void)previous_converged(a, sRed);
}

// NT: the list is read past the caches (see PS_STREAM_BYTES).
template <bool NT>
__device__ __forceinline__ uint4 load_quad(const uint4* p) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4* q = reinterpret_cast<const u32x4*>(p);
    u32x4 x;
    if constexpr (NT) x = __builtin_nontemporal_load(q);
    else x = *q;
    return make_uint4(x.x, x.y, x.z, x.w);
}

template <bool NT, bool PAIR>
__global__ __launch_bounds__(PS_WG) void k_pr_stream(StreamArgs a) {
    __shared__ __attribute__((aligned(16))) float sHub[PS_HUBS];
    __shared__ double sRed[PS_WG / WAVE];
    if (a.ctl->done) return;
    if (a.it > 1 && previous_converged(a, sRed)) return;
    {
        const float4* src = reinterpret_cast<const float4*>(a.c_old);
        float4* dst = reinterpret_cast<float4*>(sHub);
        const uint32_t quads = PAIR ? (a.hubs + 1) / 2 : a.hubs / 4;
        for (uint32_t i = threadIdx.x; i < quads; i += PS_WG) dst[i] = src[i];
    }
    __syncthreads();
    const uint32_t lane = (uint32_t)lane_id();
    const uint32_t nw = gridDim.x * (PS_WG / WAVE);
    // consecutive tiles go to different workgroups, so a remainder spreads over all CUs
    uint32_t t = (threadIdx.x / WAVE) * gridDim.x + blockIdx.x;
    if (t >= a.ntiles) return;
    // the next tile's sources are loaded while the current tile's contributions arrive
    uint4 q[PS_EPL / 4];
#pragma unroll
    for (int k = 0; k < PS_EPL / 4; ++k) q[k] = load_quad<NT>(a.tcol + ((uint64_t)t * (PS_EPL / 4) + k) * WAVE + lane);
    uint32_t d = a.desc[(uint64_t)t * WAVE + lane];
    while (true) {
        float v[PS_EPL], vl[PS_EPL];  // vl: low words of pairs
        // a hub's lane reads the hub from LDS and contribution 0 from memory (one shared line
        // per wave, dropped); branch-free, so all 16 gathers are in flight
#pragma unroll
        for (int k = 0; k < PS_EPL / 4; ++k) {
            const uint32_t u[4] = {q[k].x, q[k].y, q[k].z, q[k].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                vl[4 * k + j] = 0.0f;
                if constexpr (PAIR) {
                    const float2 h = reinterpret_cast<const float2*>(sHub)[u[j]];
                    v[4 * k + j] = h.x;
                    vl[4 * k + j] = h.y;
                    continue;
                }
                const bool hub = u[j] < a.hubs;
                const float g = a.c_old[hub ? 0u : u[j]];
                const float h = sHub[hub ? u[j] : 0u];
                v[4 * k + j] = hub ? h : g;
            }
        }
        const uint32_t ends = d & 0xffffu, row0 = a.tfirst[t] + (d >> 16);
        const uint32_t cur = t;
        t += nw;
        if (t < a.ntiles) {
#pragma unroll
            for (int k = 0; k < PS_EPL / 4; ++k) q[k] = load_quad<NT>(a.tcol + ((uint64_t)t * (PS_EPL / 4) + k) * WAVE + lane);
            d = a.desc[(uint64_t)t * WAVE + lane];
        }
        const uint64_t has = __ballot(ends != 0);
        Comp acc{0.0f, 0.0f}, first{0.0f, 0.0f};
        if (has == 0) {  // inside one row
#pragma unroll
            for (int j = 0; j < PS_EPL; ++j) acc = comp_add(acc, Comp{v[j], vl[j]});
        } else {
            uint32_t row = row0;
#pragma unroll
            for (int j = 0; j < PS_EPL; ++j) {
                acc = comp_add(acc, Comp{v[j], vl[j]});
                if ((ends >> j) & 1u) {
                    if (row == row0) first = acc;  // waits for what earlier lanes hold of the row
                    else a.sums[row] = make_float2(acc.s, acc.e);
                    ++row;
                    acc = Comp{0.0f, 0.0f};
                }
            }
        }
        // open sums scanned over the lanes since the last lane with a row end
        const uint64_t upto = has & (lanemask_lt() | (1ull << lane));
        const int from = upto ? 63 - __clzll((long long)upto) : 0;
#pragma unroll
        for (int off = 1; off < WAVE; off <<= 1) {
            Comp o;
            o.s = __shfl_up(acc.s, off, WAVE);
            o.e = __shfl_up(acc.e, off, WAVE);
            if ((int)lane - off >= from) acc = comp_add(o, acc);
        }
        Comp carry;
        carry.s = __shfl_up(acc.s, 1, WAVE);
        carry.e = __shfl_up(acc.e, 1, WAVE);
        if (ends) {
            if (lane) first = comp_add(carry, first);
            a.sums[row0] = make_float2(first.s, first.e);
        }
        if (lane == WAVE - 1) a.tail[cur] = make_float2(acc.s, acc.e);
        if (t >= a.ntiles) break;
    }
}

constexpr uint32_t PS_SPANS = 0x80000000u;  // entry flag: the row crosses wave tiles

struct FinishArgs {
    PullArgs p;                 // rank buffers, degrees, teleport terms, in-edge rows
    const uint32_t* ent;        // vertices with in-edges in vlist order | PS_SPANS
    const float2* sums;
    const float2* tail;
    const uint32_t* span;       // rows crossing at most FIX_LONG tiles, then those crossing more
    uint32_t nspan;
    const uint32_t* span_long;
    uint32_t nlong;
    uint32_t n;
    double* parts;
    float* cerr;                // per vertex: rounding error of its last contribution (no pairs)
};

// Contribution x / d of a vertex of rank x = hi + lo and out-degree d.
template <bool PAIR>
__device__ __forceinline__ void store_contribution(const FinishArgs& f, uint32_t v, double x, uint32_t d, bool feed) {
    if constexpr (PAIR) {
        const double y = d ? x / (double)d : 0.0;
        const float h = (float)y;
        reinterpret_cast<float2*>(f.p.c_new)[v] = make_float2(h, (float)(y - (double)h));
    } else {
        double y = d ? x / (double)d : 0.0;
        if (feed) y += (double)f.cerr[v];
        const float h = (float)y;
        f.p.c_new[v] = h;
        f.cerr[v] = (float)(y - (double)h);
    }
}

template <bool PAIR>
__device__ __forceinline__ void finish_row(const FinishArgs& f, uint32_t v, Comp sum, bool feed, double& res) {
    const PullArgs& a = f.p;
    const double xo = (double)a.x_old[v] + (double)a.xl_old[v];
    const uint32_t d = a.outdeg[v];
    float hi, lo;
    rank_pair(v == a.pers ? a.pers_base : a.base, a.damping, sum, &hi, &lo);
    a.x_new[v] = hi;
    a.xl_new[v] = lo;
    const double x = (double)hi + (double)lo;
    store_contribution<PAIR>(f, v, x, d, feed);
    res += fabs(x - xo);
}

// Ranks from the row sums: a thread per row; rows that cross tiles add the tails of the tiles
// they leave open in tile order (a wave per row when they are many: lane-strided, then a fixed
// tree).  Streams ~44 B per row.  Vertices without in-edges hold their teleport term from the
// first iteration on; the two buffers get it in iterations 1 and 2.
template <bool PAIR>
__global__ __launch_bounds__(WG) void k_pr_finish(FinishArgs f) {
    __shared__ double sRed[WG / WAVE];
    const PullArgs& a = f.p;
    if (a.ctl->done) return;
    // (the errors start at the second contribution; the residual of the iteration before is known)
    const bool feed = !PAIR && a.it > 1 && a.ctl->residual[(a.it - 1) & 3] > PS_FEED;
    double res = 0.0;
    const uint32_t tid = blockIdx.x * WG + threadIdx.x, nt = gridDim.x * WG;
    for (uint64_t i = tid; i < a.nz; i += nt) {
        const uint32_t v = f.ent[i];
        if (v & PS_SPANS) continue;
        const float2 s = f.sums[i];
        finish_row<PAIR>(f, v, Comp{s.x, s.y}, feed, res);
    }
    for (uint32_t i = tid; i < f.nspan; i += nt) {
        const uint32_t pos = f.span[i], v = f.ent[pos] & ~PS_SPANS;
        const uint32_t ta = (uint32_t)(a.row[v] / PS_TILE), tb = (uint32_t)((a.row[v + 1] - 1) / PS_TILE);
        Comp acc{0.0f, 0.0f};
        for (uint32_t t = ta; t < tb; ++t) acc = comp_add(acc, Comp{f.tail[t].x, f.tail[t].y});
        acc = comp_add(acc, Comp{f.sums[pos].x, f.sums[pos].y});
        finish_row<PAIR>(f, v, acc, feed, res);
    }
    const uint32_t lane = (uint32_t)lane_id();
    for (uint32_t j = tid / WAVE; j < f.nlong; j += nt / WAVE) {
        const uint32_t pos = f.span_long[j], v = f.ent[pos] & ~PS_SPANS;
        const uint32_t ta = (uint32_t)(a.row[v] / PS_TILE), tb = (uint32_t)((a.row[v + 1] - 1) / PS_TILE);
        Comp acc{0.0f, 0.0f};
        for (uint32_t t = ta + lane; t < tb; t += WAVE) acc = comp_add(acc, Comp{f.tail[t].x, f.tail[t].y});
#pragma unroll
        for (int off = WAVE / 2; off > 0; off >>= 1) {
            Comp o;
            o.s = __shfl_down(acc.s, off, WAVE);
            o.e = __shfl_down(acc.e, off, WAVE);
            acc = comp_add(acc, o);
        }
        if (lane == 0) {
            acc = comp_add(acc, Comp{f.sums[pos].x, f.sums[pos].y});
            finish_row<PAIR>(f, v, acc, feed, res);
        }
    }
    if (a.it <= 2) {
        for (uint64_t v = tid; v < f.n; v += nt) {
            if (a.row[v + 1] != a.row[v]) continue;
            const float base = (v == a.pers) ? a.pers_base : a.base;
            const double xo = (double)a.x_old[v] + (double)a.xl_old[v];
            a.x_new[v] = base;
            a.xl_new[v] = 0.0f;
            store_contribution<PAIR>(f, (uint32_t)v, (double)base, a.outdeg[v], false);
            res += fabs((double)base - xo);
        }
    }
    res = wave_sum(res);
    if (lane == 0) sRed[threadIdx.x / WAVE] = res;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int i = 0; i < WG / WAVE; ++i) t += sRed[i];
        f.parts[blockIdx.x] = t;
    }
}

// Tables of k_pr_stream, from the in-edge CSR and its list of rows (vertices with in-edges).
// desc starts as zeros; a row's last edge e sets bit e % 16 of its lane's word.
__global__ void k_ps_rows(const uint64_t* __restrict__ row, const uint32_t* __restrict__ vlist, uint32_t nz,
                          uint32_t* __restrict__ desc, uint32_t* __restrict__ ent, uint32_t* __restrict__ span,
                          uint32_t cap, uint32_t* __restrict__ count) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nz;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t v = vlist[i];
        const uint64_t last = row[v + 1] - 1;
        atomicOr(&desc[last / PS_EPL], 1u << (last % PS_EPL));
        const uint32_t ta = (uint32_t)(row[v] / PS_TILE), tb = (uint32_t)(last / PS_TILE);
        ent[i] = v | (ta != tb ? PS_SPANS : 0u);
        if (ta == tb) continue;
        if (tb - ta + 1 > FIX_LONG) span[cap - 1 - atomicAdd(&count[1], 1u)] = (uint32_t)i;
        else span[atomicAdd(&count[0], 1u)] = (uint32_t)i;
    }
}
// Per tile: the row of its first edge, and row ends before each lane.  A wave per tile.
__global__ __launch_bounds__(WG) void k_ps_tiles(const uint64_t* __restrict__ row, const uint32_t* __restrict__ vlist,
                                                 uint32_t nz, uint32_t ntiles, uint32_t* __restrict__ desc,
                                                 uint32_t* __restrict__ tfirst) {
    const uint32_t lane = (uint32_t)lane_id();
    const uint32_t nw = gridDim.x * (WG / WAVE);
    for (uint32_t t = blockIdx.x * (WG / WAVE) + threadIdx.x / WAVE; t < ntiles; t += nw) {
        const uint64_t o = (uint64_t)t * WAVE + lane;
        const uint32_t ends = desc[o] & 0xffffu;
        const uint32_t cnt = (uint32_t)__popc(ends);
        desc[o] = ends | ((wave_incl_scan(cnt) - cnt) << 16);
        if (lane == 0) {
            const uint64_t e = (uint64_t)t * PS_TILE;
            uint32_t lo = 0, hi = nz;  // last row that starts at or before e
            while (hi - lo > 1) {
                const uint32_t mid = lo + (hi - lo) / 2;
                if (row[vlist[mid]] <= e) lo = mid; else hi = mid;
            }
            tfirst[t] = lo;
        }
    }
}
// out[tile][k][lane] = edges 4k .. 4k+3 of that lane's 16 (source 0 past the last edge)
__global__ void k_ps_layout(const uint32_t* __restrict__ col, uint64_t m, uint64_t quads, uint4* __restrict__ out) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < quads;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t tile = i / (PS_TILE / 4), r = i % (PS_TILE / 4), k = r / WAVE, lane = r % WAVE;
        const uint64_t e = tile * PS_TILE + lane * PS_EPL + 4 * k;
        uint4 x = make_uint4(0, 0, 0, 0);
        if (e + 4 <= m) {
            x = *reinterpret_cast<const uint4*>(col + e);
        } else {
            if (e < m) x.x = col[e];
            if (e + 1 < m) x.y = col[e + 1];
            if (e + 2 < m) x.z = col[e + 2];
        }
        out[i] = x;
    }
}

}  // namespace

// Tables of the streamed gather, built once per graph (the rows do not depend on K).  Called
// with the graph's lock held or before concurrent queries start, after ensure_tigr(in, K).
// Leaves ps.built false where they do not fit in memory or vertex ids need 32 bits: the sync
// variants then run the pull.
static eeg_status ensure_pr_stream(eeg_graph* g, uint32_t K) {
    PrStream& ps = g->prstream;
    if (ps.built || ps.refused) return EEG_OK;
    const Tigr& t = g->tin[k_index(K)];
    const Csr& in = g->in;
    ps.refused = true;
    if (g->n >= PS_SPANS || t.nz == 0) return EEG_OK;
    const uint64_t ntiles = (in.m + PS_TILE - 1) / PS_TILE;
    const uint32_t cap = (uint32_t)ntiles + 1;
    DevMem cnt;
    if (ps.tcol.alloc(ntiles * PS_TILE * 4) != EEG_OK || ps.desc.alloc(ntiles * WAVE * 4) != EEG_OK ||
        ps.tfirst.alloc(ntiles * 4) != EEG_OK || ps.ent.alloc((size_t)t.nz * 4) != EEG_OK ||
        ps.span.alloc((size_t)cap * 4) != EEG_OK || cnt.alloc(8) != EEG_OK) {
        clear_error();
        for (DevMem* d : {&ps.tcol, &ps.desc, &ps.tfirst, &ps.ent, &ps.span}) d->release();
        return EEG_OK;
    }
    hipStream_t s = g->stream;
    auto grid = [](uint64_t work) { return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(16384, (work + WG - 1) / WG)); };
    EEG_HIP(hipMemsetAsync(ps.desc.p, 0, ntiles * WAVE * 4, s));
    EEG_HIP(hipMemsetAsync(cnt.p, 0, 8, s));
    k_ps_rows<<<grid(t.nz), WG, 0, s>>>(in.rowp(), t.vlist.as<uint32_t>(), t.nz, ps.desc.as<uint32_t>(),
                                        ps.ent.as<uint32_t>(), ps.span.as<uint32_t>(), cap, cnt.as<uint32_t>());
    k_ps_tiles<<<grid(ntiles * WAVE), WG, 0, s>>>(in.rowp(), t.vlist.as<uint32_t>(), t.nz, (uint32_t)ntiles,
                                                  ps.desc.as<uint32_t>(), ps.tfirst.as<uint32_t>());
    k_ps_layout<<<grid(ntiles * (PS_TILE / 4)), WG, 0, s>>>(in.colp(), in.m, ntiles * (PS_TILE / 4), ps.tcol.as<uint4>());
    EEG_HIP(hipGetLastError());
    uint32_t ns[2] = {0, 0};
    EEG_HIP(hipMemcpyAsync(ns, cnt.p, 8, hipMemcpyDeviceToHost, s));
    EEG_HIP(hipStreamSynchronize(s));
    if ((uint64_t)ns[0] + ns[1] > cap) return fail(EEG_ERR_DEVICE, "PageRank span list overflow");
    ps.nspan = ns[0];
    ps.nlong = ns[1];
    ps.span_cap = cap;
    ps.ntiles = (uint32_t)ntiles;
    ps.nz = t.nz;
    ps.refused = false;
    ps.built = true;
    return EEG_OK;
}

// Tables of the PageRank gathers: the streamed one's, or where it is not available and for the
// in-place sweeps the vertices of the in-edge Tigr table whose virtual nodes cross a pull tile,
// listed once per graph and K (their partial sums are combined by k_pr_fix).  Called with the
// graph's lock held or before concurrent queries start.
eeg_status ensure_pr_span(eeg_graph* g, uint32_t K, bool inplace) {
    Tigr& t = g->tin[k_index(K)];
    if (!g->outdeg.p) {  // out-degrees as u32, read by every PageRank iteration
        EEG_TRY(g->outdeg.alloc((size_t)g->n * 4 + 4));
        if (g->n) {
            k_outdeg<<<std::max(1u, std::min(8192u, (g->n + WG - 1) / WG)), WG, 0, g->stream>>>(
                g->out.rowp(), g->n, g->outdeg.as<uint32_t>());
            EEG_HIP(hipGetLastError());
        }
    }
    // (the pull's tables are small; their memory is taken first, so that it can always run)
    const uint32_t TV = PR_TILE / K;
    const uint64_t ntiles = (t.P + TV - 1) / TV;
    const uint32_t cap = (uint32_t)ntiles + 1;
    EEG_TRY(t.span.alloc((size_t)cap * 4 + 8));  // and two counters
    EEG_TRY(t.prstart.alloc((size_t)ntiles * 4 + 4));
    if (!inplace) {
        EEG_TRY(ensure_pr_stream(g, K));
        if (g->prstream.built) return EEG_OK;
    }
    if (t.span_built) return EEG_OK;
    hipStream_t s = g->stream;
    uint32_t* cnt = t.span.as<uint32_t>() + cap;
    EEG_HIP(hipMemsetAsync(cnt, 0, 8, s));
    if (t.nz) {
        k_list_spanning<<<std::max(1u, std::min(8192u, (t.nz + WG - 1) / WG)), WG, 0, s>>>(
            t.vscan.as<uint32_t>(), t.nz, TV, cap, t.span.as<uint32_t>(), cnt);
        EEG_HIP(hipGetLastError());
        k_tile_starts<<<std::max<uint64_t>(1, std::min<uint64_t>(4096, (ntiles + WG - 1) / WG)), WG, 0, s>>>(
            t.vscan.as<uint32_t>(), t.nz, TV, (uint32_t)ntiles, t.prstart.as<uint32_t>());
        EEG_HIP(hipGetLastError());
    }
    uint32_t ns[2] = {0, 0};
    EEG_HIP(hipMemcpyAsync(ns, cnt, 8, hipMemcpyDeviceToHost, s));
    EEG_HIP(hipStreamSynchronize(s));
    if ((uint64_t)ns[0] + ns[1] > cap) return fail(EEG_ERR_DEVICE, "PageRank span list overflow");
    t.nspan = ns[0];
    t.nspan_long = ns[1];
    t.span_cap = cap;
    t.span_built = true;
    return EEG_OK;
}

eeg_status run_pagerank(eeg_graph* g, uint32_t algo, uint32_t source, const eeg_opts& o,
                        eeg_stats* st, Work* wk, hipStream_t sk) {
    const auto t_host0 = std::chrono::steady_clock::now();
    const bool personalised = (algo == EEG_PPR);
    // async variants update ranks in place (Gauss-Seidel in tile order): a gather may see a
    // neighbour's rank of this sweep or of the last one, so the sum order is not fixed, but the
    // iteration converges in fewer sweeps and needs no atomics
    const bool inplace = (o.variant == EEG_ASYNC_PUSH_TD || o.variant == EEG_ASYNC_PUSH_DD);
    const uint32_t K = o.K ? o.K : 8;
    if (k_index(K) < 0) return fail(EEG_ERR_INVALID_ARG, "K must be 4, 8, 16 or 32 (got %u)", K);
    const float d = o.damping > 0 ? o.damping : 0.85f;
    if (!(d > 0 && d < 1)) return fail(EEG_ERR_INVALID_ARG, "damping must be in (0,1)");
    const double eps = o.epsilon > 0 ? o.epsilon : 1e-7;
    const uint32_t max_iters = o.max_iters ? o.max_iters : 10000;
    const uint32_t n = g->n;
    hipStream_t s = wk ? sk : g->stream;
    Work& w = wk ? *wk : g->work;
    EEG_TRY(ensure_in(g));
    EEG_TRY(ensure_tigr(g, g->in, g->tin, K));
    const Tigr& t = g->tin[k_index(K)];
    const PrStream& ps = g->prstream;
    const uint32_t TV = PR_TILE / K;
    const uint64_t pull_tiles = (t.P + TV - 1) / TV;
    int cus = 256;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, g->device);
    // workgroups per CU: more than stay resident (8), so tiles are handed out as workgroups
    // finish; 48 for the Jacobi gather, 24 in place (whose sweep count also depends on it)
    const uint32_t wpc = o.wgs_per_cu ? o.wgs_per_cu : (inplace ? 24u : 48u);
    const unsigned grid_pull = (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(pull_tiles, (uint64_t)cus * wpc));
    const unsigned grid_iso = std::max(1u, std::min(4096u, (n + WG - 1) / WG));
    constexpr unsigned FIX_WGS = 1024;

    // What the pull needs comes first: the streamed gather's tables and buffers take memory that is
    // left over, and where there is too little of it the pull runs.
    auto pull_state = [&]() -> eeg_status {
        EEG_TRY(w.ctl.alloc(sizeof(Ctl)));
        if (!w.host_ctl) EEG_HIP(hipHostMalloc((void**)&w.host_ctl, 2 * sizeof(Ctl), hipHostMallocDefault));
        for (int i = 0; i < 2; ++i) {
            EEG_TRY(w.fx[i].alloc((size_t)n * 4 + 4));
            EEG_TRY(w.fc[i].alloc((size_t)n * (n <= PS_PAIRS ? 8 : 4) + 8));
            EEG_TRY(w.fl[i].alloc((size_t)n * 4 + 4));
        }
        EEG_TRY(w.spill.alloc((size_t)(pull_tiles + 1) * 2 * sizeof(float2)));
        EEG_TRY(w.red.alloc((size_t)std::max(grid_pull + FIX_WGS + grid_iso, PS_PARTS) * sizeof(double)));
        return w.lab.alloc((size_t)n * 4 + 4);
    };
    EEG_TRY(pull_state());
    EEG_TRY(ensure_pr_span(g, K, inplace));
    bool stream = !inplace && ps.built;
    if (stream) {
        auto stream_state = [&]() -> eeg_status {
            EEG_TRY(w.spill.alloc((size_t)(ps.ntiles + 1) * 2 * sizeof(float2)));
            EEG_TRY(w.psum.alloc((size_t)ps.nz * sizeof(float2)));
            return n > PS_PAIRS ? w.cerr.alloc((size_t)n * 4) : EEG_OK;
        };
        const eeg_status got = stream_state();
        if (got == EEG_ERR_OOM) {
            clear_error();
            stream = false;
            EEG_TRY(pull_state());
            std::unique_lock<std::mutex> lk(g->mu, std::defer_lock);
            if (wk) lk.lock();  // (otherwise the caller holds it)
            EEG_TRY(ensure_pr_span(g, K, true));
        } else {
            EEG_TRY(got);
        }
    }
    const bool pairs = stream && n <= PS_PAIRS;
    const uint64_t ntiles = stream ? ps.ntiles : pull_tiles;
    if (!stream && w.cerr.alloc((size_t)n * 4) != EEG_OK) clear_error();  // the pull does without
    // vertices whose virtual nodes cross a tile boundary (finished by k_pr_fix)
    const DevMem& span = t.span;
    const uint32_t nshort = t.nspan, nlong = t.nspan_long;
    const uint32_t nspan = nshort + nlong;
    const uint32_t* span_long = span.as<uint32_t>() + (t.span_cap - nlong);
    // the fix-up order only matters within a vertex, so the list order is irrelevant

    const unsigned grid_fix = std::max(1u, std::min(FIX_WGS, std::max((nshort + WG - 1) / WG, (nlong + 3) / 4)));
    // streamed gather: its LDS admits one workgroup of 1024 threads per CU, which keeps its hubs
    // for all its tiles; a given wgs_per_cu counts 256-thread workgroups, so more take turns (a
    // serving lane leaves gaps for others).  At least 4 tiles per workgroup, and no more hubs
    // than the workgroup has edges, so copying them stays below what they save.
    const unsigned grid_stream = (unsigned)std::max<uint64_t>(
        1, std::min<uint64_t>((ntiles + 3) / 4, (uint64_t)cus * (o.wgs_per_cu ? (o.wgs_per_cu + 3) / 4 : 1)));
    const unsigned grid_finish = std::max(1u, std::min(PS_PARTS, (n + WG - 1) / WG));
    const uint32_t nparts = stream ? grid_finish : grid_pull + grid_fix + grid_iso;
    EEG_HIP(hipMemsetAsync(w.red.p, 0, (size_t)nparts * sizeof(double), s));

    Ctl* ctl = w.ctl.as<Ctl>();
    EEG_HIP(hipMemsetAsync(ctl, 0, sizeof(Ctl), s));
    const float x0 = 1.0f / (float)n;
    const float base = personalised ? 0.0f : (1.0f - d) / (float)n;
    const uint32_t pers = personalised ? source : 0xffffffffu;
    (pairs ? k_pr_init<true> : k_pr_init<false>)<<<grid_iso, WG, 0, s>>>(
        g->outdeg.as<uint32_t>(), n, x0, pers, w.fx[0].as<float>(), w.fl[0].as<float>(), w.fc[0].as<float>());
    EEG_HIP(hipGetLastError());

    PullArgs pa{};
    pa.row = g->in.rowp();
    pa.col = g->in.colp();
    pa.vlist = t.vlist.as<uint32_t>();
    pa.vscan = t.vscan.as<uint32_t>();
    pa.nz = t.nz;
    pa.P = (uint32_t)t.P;
    pa.outdeg = g->outdeg.as<uint32_t>();
    pa.spill = w.spill.as<float2>();
    pa.ctl = ctl;
    pa.base = base;
    pa.damping = d;
    pa.pers = pers;
    pa.pers_base = 1.0f - d;
    pa.strided = inplace ? 1u : 0u;
    pa.tstart = t.prstart.as<uint32_t>();
    double* red = w.red.as<double>();
    auto pull_fn = (K == 4) ? k_pr_pull<4, false> : (K == 8) ? k_pr_pull<8, false>
                   : (K == 16) ? k_pr_pull<16, false> : k_pr_pull<32, false>;
    auto pull_feed_fn = (K == 4) ? k_pr_pull<4, true> : (K == 8) ? k_pr_pull<8, true>
                        : (K == 16) ? k_pr_pull<16, true> : k_pr_pull<32, true>;
    bool feed = false;  // the pull has been seen to want its rounding errors fed back

    const bool nontemporal = (uint64_t)ps.ntiles * PS_TILE * 4 > PS_STREAM_BYTES;
    StreamArgs sa{};
    FinishArgs fa{};
    if (stream) {
        sa.tcol = ps.tcol.as<uint4>();
        sa.desc = ps.desc.as<uint32_t>();
        sa.tfirst = ps.tfirst.as<uint32_t>();
        sa.ntiles = ps.ntiles;
        sa.hubs = pairs ? n : (uint32_t)std::min<uint64_t>(std::min(n, PS_HUBS), ntiles * PS_TILE / grid_stream) & ~3u;
        sa.sums = w.psum.as<float2>();
        sa.tail = w.spill.as<float2>();
        sa.parts = red;
        sa.nparts = nparts;
        sa.eps = eps;
        sa.ctl = ctl;
        fa.ent = ps.ent.as<uint32_t>();
        fa.sums = w.psum.as<float2>();
        fa.tail = w.spill.as<float2>();
        fa.span = ps.span.as<uint32_t>();
        fa.nspan = ps.nspan;
        fa.span_long = ps.span.as<uint32_t>() + (ps.span_cap - ps.nlong);
        fa.nlong = ps.nlong;
        fa.n = n;
        fa.parts = red;
        fa.cerr = w.cerr.as<float>();
    }

    hipEvent_t ev_start;
    EEG_TRY(w.event(0, &ev_start));
    // a timing event after iteration `it` is recorded only where the run may end (the last
    // iteration of every chunk and the iterations near the predicted end): each record costs
    // device time between the launches
    std::vector<uint8_t> recorded;
    uint32_t predicted_end = 0xffffffffu;
    auto launch = [&](uint32_t it, bool rec) -> eeg_status {
        pa.it = it;
        const int ob = inplace ? 0 : (int)((it - 1) & 1), nb = inplace ? 0 : (int)(it & 1);
        pa.x_old = w.fx[ob].as<float>();
        pa.xl_old = w.fl[ob].as<float>();
        pa.c_old = w.fc[ob].as<float>();
        pa.x_new = w.fx[nb].as<float>();
        pa.xl_new = w.fl[nb].as<float>();
        pa.c_new = w.fc[nb].as<float>();
        pa.res_part = red;
        hipEvent_t eb, ea;
        if (o.timing) {
            EEG_TRY(w.event(2 * (size_t)it - 1, &eb));
            EEG_HIP(hipEventRecord(eb, s));
        }
        if (stream) {
            sa.c_old = pa.c_old;
            sa.it = it;
            (nontemporal ? (pairs ? k_pr_stream<true, true> : k_pr_stream<true, false>)
                         : (pairs ? k_pr_stream<false, true> : k_pr_stream<false, false>))<<<grid_stream, PS_WG, 0, s>>>(sa);
            fa.p = pa;
            (pairs ? k_pr_finish<true> : k_pr_finish<false>)<<<grid_finish, WG, 0, s>>>(fa);
            EEG_HIP(hipGetLastError());
        } else if (t.P) {
            pa.cerr = feed ? w.cerr.as<float>() : nullptr;
            void* args[] = {&pa};
            EEG_HIP(hipLaunchKernel((const void*)(feed ? pull_feed_fn : pull_fn), dim3(grid_pull), dim3(WG), args, 0, s));
        } else {
            EEG_HIP(hipMemsetAsync(red, 0, grid_pull * sizeof(double), s));
        }
        if (!stream && nspan) {
            k_pr_fix<<<grid_fix, WG, 0, s>>>(pa, span.as<uint32_t>(), nshort, span_long, nlong, TV,
                                             red + grid_pull);
            EEG_HIP(hipGetLastError());
        }
        const uint32_t iso_iters = inplace ? 1 : 2;  // vertices without in-edges settle at once
        if (!stream && it <= iso_iters) {
            k_pr_isolated<<<grid_iso, WG, 0, s>>>(g->in.rowp(), g->outdeg.as<uint32_t>(), n, pa.x_old, pa.xl_old,
                                                  pa.x_new, pa.xl_new, pa.c_new, base, pers, 1.0f - d,
                                                  red + grid_pull + grid_fix, ctl);
            EEG_HIP(hipGetLastError());
        } else if (!stream && it == iso_iters + 1) {
            EEG_HIP(hipMemsetAsync(red + grid_pull + grid_fix, 0, grid_iso * sizeof(double), s));
        }
        // (the streamed gather sums the residual at the start of the next iteration)
        if (!stream) k_pr_reduce<<<1, RED_WG, 0, s>>>(red, nparts, ctl, it, eps, FeedRule(d), feed);
        EEG_HIP(hipGetLastError());
        if (recorded.size() <= it) recorded.resize((size_t)it + 64, 0);
        recorded[it] = (rec || o.timing) ? 1 : 0;
        if (recorded[it]) {
            hipEvent_t ea2;
            EEG_TRY(w.event(2 * (size_t)it, &ea2));
            EEG_HIP(hipEventRecord(ea2, s));
        }
        (void)ea;
        return EEG_OK;
    };
    if (!stream && !nspan) EEG_HIP(hipMemsetAsync(red + grid_pull, 0, grid_fix * sizeof(double), s));

    EEG_HIP(hipEventRecord(ev_start, s));
    uint32_t it = 1;
    eeg_status rc = EEG_OK;
    {
        uint32_t chunk = 4;
        EEG_TRY(w.poll_events());
        hipEvent_t* poll = w.poll;
        bool pending[2] = {false, false};  // a copy of this run is in flight in the slot
        // queues up to `chunk` iterations, never past max_iters (callers check it <= max_iters)
        auto submit = [&](int slot) -> eeg_status {
            const uint32_t cnt = std::min<uint32_t>(chunk, max_iters + 1 - it);
            for (uint32_t k = 0; k < cnt; ++k, ++it)
                EEG_TRY(launch(it, k + 1 == cnt || (predicted_end != 0xffffffffu && it + 2 >= predicted_end)));
            if (stream) {
                sa.it = it;
                k_pr_check<<<1, PS_WG, 0, s>>>(sa);
                EEG_HIP(hipGetLastError());
            }
            EEG_HIP(hipMemcpyAsync(&w.host_ctl[slot], ctl, sizeof(Ctl), hipMemcpyDeviceToHost, s));
            EEG_HIP(hipEventRecord(poll[slot], s));
            pending[slot] = true;
            chunk = std::min<uint32_t>(chunk * 2, 16);
            return EEG_OK;
        };
        // Iterations still needed after the polled one: the residual decays geometrically, so
        // log(eps / r_k) / log(r_k / r_k-1) (16 when the last two residuals do not show it).
        auto remaining = [&](const Ctl& h) -> uint32_t {
            const uint32_t k = h.iters;
            if (k < 2) return 16;
            const double r1 = h.residual[k & 3], r0 = h.residual[(k - 1) & 3];
            if (!(r1 > 0.0) || !(r0 > r1)) return 16;
            const double need = std::log(eps / r1) / std::log(r1 / r0);
            return need < 1.0 ? 1u : (uint32_t)std::min(16.0, std::ceil(need));
        };
        int cur = 0;
        rc = submit(0);
        while (rc == EEG_OK) {
            if (it <= max_iters) rc = submit(cur ^ 1);
            if (rc != EEG_OK) break;
            EEG_HIP(hipEventSynchronize(poll[cur]));
            pending[cur] = false;
            const Ctl& h = w.host_ctl[cur];
            if (h.done) break;
            if (!pending[cur ^ 1]) {  // max_iters launched and none of them converged
                rc = fail(EEG_ERR_NOT_CONVERGED, "PageRank residual above %g after %u iterations", eps, max_iters);
                break;
            }
            // size the next chunk to the predicted remainder beyond what is in flight (+1), so
            // few launches run after convergence; a short prediction costs one more poll
            const uint32_t inflight = (it - 1) - h.iters, rem = remaining(h);
            chunk = rem > inflight ? std::min<uint32_t>(rem - inflight + 1, 16) : 1u;
            predicted_end = h.iters + rem;
            feed = feed || (h.feed && w.cerr.p && !stream);
            cur ^= 1;
        }
    }
    EEG_HIP(hipStreamSynchronize(s));
    EEG_HIP(hipMemcpy(w.host_ctl, ctl, sizeof(Ctl), hipMemcpyDeviceToHost));
    const Ctl hc = w.host_ctl[0];
    const uint32_t iters = hc.iters;
    if (rc == EEG_OK && !hc.done)
        rc = fail(EEG_ERR_NOT_CONVERGED, "PageRank residual above %g after %u iterations", eps, max_iters);
    // result: the buffer written by the last iteration, copied into the label slot
    const int fb = inplace ? 0 : (int)(iters & 1);
    k_pr_output<<<grid_iso, WG, 0, s>>>(w.fx[fb].as<float>(), w.fl[fb].as<float>(), n, w.lab.as<float>());
    EEG_HIP(hipGetLastError());
    EEG_HIP(hipStreamSynchronize(s));
    if (st) {
        // the first recorded event at or after the last working iteration (every chunk ends
        // with one, so at worst a few no-op launches past it)
        uint32_t ie = std::max<uint32_t>(iters, 1);
        while (ie < recorded.size() && !recorded[ie]) ++ie;
        if (ie >= recorded.size()) ie = (uint32_t)recorded.size() - 1;
        hipEvent_t ev_end;
        EEG_TRY(w.event(2 * (size_t)ie, &ev_end));
        float ms = 0;
        EEG_HIP(hipEventElapsedTime(&ms, ev_start, ev_end));
        st->iterations = iters;
        st->launches = it - 1;
        st->ms_traversal = ms;
        st->pr_residual = hc.residual[iters & 3];
        st->edges_relaxed = (uint64_t)iters * g->m;
        st->vertices_touched = (uint64_t)iters * n;
        // per iteration: 4 B source index + 4 B contribution per in-edge and 8 B per vertex
        // (rank read and write); the row offsets, out-degrees, second rank word and
        // contributions this layout also moves (32 B more per vertex) are not counted
        st->bytes_alg = (double)iters * (8.0 * (double)g->m + 8.0 * (double)n);
        double ksum = 0;
        uint32_t kn = 0;
        if (o.timing) {
            for (uint32_t i = 1; i <= iters; ++i) {
                hipEvent_t eb, ea;
                EEG_TRY(w.event(2 * (size_t)i - 1, &eb));
                EEG_TRY(w.event(2 * (size_t)i, &ea));
                float km = 0;
                EEG_HIP(hipEventElapsedTime(&km, eb, ea));
                ksum += km;
                ++kn;
            }
        }
        st->ms_kernel_sum = ksum;
        st->kernels_timed = kn;
        st->ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_host0).count();
    }
    return rc;
}


}  // namespace eeg
