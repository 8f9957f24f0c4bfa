// Sorted frontier queues, shared by the single-query traversals (relax.hip) and the batched
// plane passes (batch.hip): a kernel that improved a vertex marks it (a byte per vertex and a byte
// per 16384 vertices), and compact_frontier turns the marks into the next queue in vertex order.
//
// Marks are bytes written by plain stores because atomics are performed past the L2 at about 24 G/s
// whatever they do: as bits set with atomicOr they were half of the atomics of a traversal
// (SSSP on the 4096^2 grid: relaxations 8.0 -> 5.3 ms).  The byte per chunk lets thin frontiers skip
// the rest: a compaction reads n / 16384 bytes and the chunks that were touched.
#pragma once

#include "device.hpp"

namespace eeg {
namespace {

// Threads and vertices of one workgroup's compaction step.  Each step ends in one atomicAdd on the
// same word, which takes its turn for about 12 ns: with 256 threads the 2048 of a 16.8 M vertex
// graph took 20 us more than these 1024 (thin frontiers over the whole 4096^2 grid: 32 -> 24 us).
constexpr int COMPACT_WG = 1024;
constexpr int COMPACT_PER = 16;  // vertices per thread
constexpr uint32_t MARK_CHUNK = COMPACT_PER * COMPACT_WG;

inline uint32_t mark_chunks(uint32_t n) { return (uint32_t)(((uint64_t)n + MARK_CHUNK - 1) / MARK_CHUNK); }
// one allocation: the vertices' bytes (whole chunks), then the chunks' bytes, as whole words
inline size_t mark_bytes(uint32_t n) {
    const size_t c = mark_chunks(n);
    return c * MARK_CHUNK + (c + 3) / 4 * 4;
}
inline uint8_t* chunk_marks(void* marks, uint32_t n) {
    return static_cast<uint8_t*>(marks) + (size_t)mark_chunks(n) * MARK_CHUNK;
}

__device__ __forceinline__ void set_mark(uint8_t* mark, uint8_t* cmark, uint32_t u) {
    mark[u] = 1;
    cmark[u / MARK_CHUNK] = 1;
}

// Sorted frontier: the vertices that iteration `it` marked, with out-edges, as the next queue
// (buffer it & 1, Ctl slot it % 3), in ascending id order within each block's 16384-vertex
// chunk; chunks take their queue ranges in the order their atomic lands.  Marks are cleared as
// they are read.  One thread per 16 vertices.
struct CompactArgs {
    uint8_t* mark;
    uint8_t* cmark;
    uint32_t n;
    const uint32_t* vnc;
    Ctl* ctl;
    uint32_t *qa, *sa, *qb, *sb;  // queue buffers 0 and 1
    uint32_t cap;
    uint32_t it;
};

// four bytes of 0 or 1 -> four bits
__device__ __forceinline__ uint32_t mark_bits(uint32_t x) { return (x * 0x10204080u) >> 28; }

// Every thread of the grid (COMPACT_WG a workgroup) calls it.
__device__ __forceinline__ void compact_frontier(const CompactArgs& a) {
    const uint32_t it = a.it;
    Ctl* ctl = a.ctl;
    uint32_t* qout = (it & 1u) ? a.qb : a.qa;
    uint32_t* sout = (it & 1u) ? a.sb : a.sa;
    const int slot = (int)(it % 3u);
    __shared__ uint64_t sScan[COMPACT_WG / WAVE + 1];
    __shared__ uint32_t sBase[2];
    const uint32_t chunks = (uint32_t)(((uint64_t)a.n + MARK_CHUNK - 1) / MARK_CHUNK);
    for (uint32_t c = blockIdx.x; c < chunks; c += gridDim.x) {
        if (!__syncthreads_or(a.cmark[c] != 0)) continue;  // the same answer in every thread
        if (threadIdx.x == 0) a.cmark[c] = 0;              // read by every thread above
        const uint32_t v0 = c * MARK_CHUNK + threadIdx.x * COMPACT_PER;
        uint4* mp = reinterpret_cast<uint4*>(a.mark + v0);
        const uint4 m = *mp;
        const uint32_t word = mark_bits(m.x) | mark_bits(m.y) << 4 | mark_bits(m.z) << 8 | mark_bits(m.w) << 12;
        // the virtual-node counts, read once as vector loads (the last vertices read only the
        // counts that exist)
        uint32_t cv[COMPACT_PER];
        if (word) {
            *mp = make_uint4(0, 0, 0, 0);
            if (v0 + COMPACT_PER <= a.n) {
                const uint4* p = reinterpret_cast<const uint4*>(a.vnc + v0);
#pragma unroll
                for (int k = 0; k < COMPACT_PER / 4; ++k) {
                    const uint4 x = p[k];
                    cv[4 * k] = x.x;
                    cv[4 * k + 1] = x.y;
                    cv[4 * k + 2] = x.z;
                    cv[4 * k + 3] = x.w;
                }
            } else {
#pragma unroll
                for (int b = 0; b < COMPACT_PER; ++b) cv[b] = (v0 + (uint32_t)b < a.n) ? a.vnc[v0 + b] : 0u;
            }
        } else {
#pragma unroll
            for (int b = 0; b < COMPACT_PER; ++b) cv[b] = 0u;
        }
        uint32_t cnt = 0, vs = 0;
#pragma unroll
        for (int b = 0; b < COMPACT_PER; ++b) {
            const bool on = ((word >> b) & 1u) && cv[b];
            cnt += on ? 1u : 0u;
            vs += on ? cv[b] : 0u;
        }
        uint64_t tot;
        const uint64_t pre = block_excl_scan<uint64_t, COMPACT_WG>(((uint64_t)vs << 32) | cnt, sScan, &tot);
        if (threadIdx.x == 0) {
            const unsigned long long old = tot ? atomicAdd(&ctl->qpack[slot], (unsigned long long)tot) : 0ull;
            sBase[0] = (uint32_t)(old & 0xffffffffull);
            sBase[1] = (uint32_t)(old >> 32);
        }
        __syncthreads();
        uint32_t e = sBase[0] + (uint32_t)(pre & 0xffffffffull);
        uint32_t vv = sBase[1] + (uint32_t)(pre >> 32);
#pragma unroll
        for (int b = 0; b < COMPACT_PER; ++b) {
            // vertices without out-edges are left out: their labels are final, nothing to push
            if (!((word >> b) & 1u) || !cv[b]) continue;
            if (e < a.cap) {
                qout[e] = v0 + (uint32_t)b;
                sout[e] = vv;
            } else {
                atomicOr(&ctl->err, 2u);
            }
            ++e;
            vv += cv[b];
        }
        __syncthreads();  // sBase is rewritten by the next chunk
    }
}

}  // namespace
}  // namespace eeg
