// Packed graphs: many independent graphs laid side by side in one HBM-resident CSR (vertex ids
// offset by the vertex counts of the graphs before them, edge rows by their edge counts), so a
// single traversal seeded with one source per graph answers every graph in one launch
// sequence.  The graphs are disjoint, so graph i's labels depend on graph i's source alone and
// equal its single-query answer bit for bit; min-label CC labels come back as union ids and
// are shifted back by the graph's vertex offset.  No counterpart exists in the reference,
// whose drivers run one graph per process (src/main.cu:101-121).
//
// The union is cached for the most recent list of graphs (by handle serial), together with its
// Tigr and symmetrised tables, so repeated calls on the same set pay the packing once.
#include <algorithm>
#include <chrono>
#include <cstring>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

#include "engine.hpp"
#include "hostcopy.hpp"

namespace eeg {
namespace {

unsigned grid_pk(uint64_t work, unsigned cap = 16384) {
    uint64_t g = (work + WG - 1) / WG;
    if (g == 0) g = 1;
    return (unsigned)(g > cap ? cap : g);
}

// One member of a union and its place there, in device memory.
struct PackMember {
    const uint64_t* row;
    const uint32_t *col, *w, *perm, *inv;
    uint64_t m, eoff;
    uint32_t n, voff;
};
// A run of at most PACK_CHUNK edges (first of them, bit 63 clear) or vertices (bit 63 set) of a
// member; the workgroups take chunks, so graphs of 2^12 and 2^20 vertices fill the chip alike.
constexpr uint32_t PACK_CHUNK = 16384;
constexpr uint64_t PACK_VERTS = 1ull << 63;
struct PackChunk {
    uint64_t first;
    uint32_t member;
    uint32_t pad;
};

// Copies the members' rows, edges and orders into the union, shifted by their offsets.  Bound by
// the 16 bytes that an edge moves; one launch for all members (five for each of 64 graphs took
// their turn at ~5 us).
__global__ __launch_bounds__(WG) void k_pack(const PackChunk* __restrict__ chunks, const PackMember* __restrict__ mem,
                                             uint64_t* __restrict__ row, uint32_t* __restrict__ col,
                                             uint32_t* __restrict__ w, uint32_t* __restrict__ perm,
                                             uint32_t* __restrict__ inv) {
    const PackChunk c = chunks[blockIdx.x];
    const PackMember g = mem[c.member];
    if (c.first & PACK_VERTS) {
        const uint64_t f = c.first & ~PACK_VERTS, e = min(f + PACK_CHUNK, (uint64_t)g.n);
        for (uint64_t v = f + threadIdx.x; v < e; v += WG) {
            row[g.voff + v] = g.row[v] + g.eoff;
            perm[g.voff + v] = g.perm[v] + g.voff;
            inv[g.voff + v] = g.inv[v] + g.voff;
        }
        // the row after the last is the next member's first, written with the same value by both
        if (e == g.n && threadIdx.x == 0) row[g.voff + e] = g.row[e] + g.eoff;
        return;
    }
    const uint64_t e = min(c.first + PACK_CHUNK, g.m);
    uint32_t* cd = col + g.eoff;
    uint32_t* wd = w + g.eoff;
#pragma unroll 4
    for (uint64_t i = c.first + threadIdx.x; i < e; i += WG) {
        cd[i] = __builtin_nontemporal_load(&g.col[i]) + g.voff;
        if (w) wd[i] = __builtin_nontemporal_load(&g.w[i]);
    }
}

struct Packed {
    std::vector<uint64_t> serials;
    std::vector<uint32_t> voff;  // ngraphs + 1 vertex offsets
    eeg_graph* g = nullptr;      // the union (no host copy of the order: members have theirs)
    DevMem seeds;
    DevMem table;                // members and chunks of the copy
    ~Packed() { delete g; }
};

// Hands an allocation of the union before to the next one, unless that needs less than a quarter
// of it (a hipFree and hipMalloc of 1 GiB take milliseconds).  Only for memory whose size is
// checked where it is used.
void carry(DevMem& from, DevMem& to, uint64_t need) {
    if (from.p && from.bytes / 4 <= need) from.swap(to);
}

std::mutex g_pack_mu;
Packed* g_pack = nullptr;  // most recent union (one at a time bounds the HBM held)

// `old`: the union before (or null), whose memory is taken over where it fits; the rest is freed
// before anything is allocated.
eeg_status build_union(eeg_graph* const* gs, uint32_t k, Packed* pk, std::unique_ptr<Packed> old) {
    uint64_t N = 0, M = 0;
    const bool weighted = gs[0]->weighted;
    pk->voff.assign(k + 1, 0);
    std::vector<PackMember> mem(k);
    std::vector<PackChunk> chunks;
    for (uint32_t i = 0; i < k; ++i) {
        const eeg_graph* gi = gs[i];
        if (gi->device != gs[0]->device) return fail(EEG_ERR_INVALID_ARG, "graphs live on different devices");
        if (gi->weighted != weighted)
            return fail(EEG_ERR_INVALID_ARG, "weighted and unweighted graphs cannot be packed together");
        pk->voff[i] = (uint32_t)N;
        mem[i] = PackMember{gi->out.rowp(), gi->out.colp(), gi->out.wp(), gi->perm.as<uint32_t>(),
                            gi->inv.as<uint32_t>(), gi->m, M, gi->n, (uint32_t)N};
        for (uint64_t f = 0; f < gi->m; f += PACK_CHUNK) chunks.push_back(PackChunk{f, i, 0});
        for (uint64_t f = 0; f < gi->n; f += PACK_CHUNK) chunks.push_back(PackChunk{f | PACK_VERTS, i, 0});
        N += gi->n;
        M += gi->m;
        if (N > 0xfffffff0ull) return fail(EEG_ERR_UNSUPPORTED, "packed vertex count exceeds 2^32 - 16");
    }
    pk->voff[k] = (uint32_t)N;
    eeg_graph* u = nullptr;
    EEG_TRY(new_graph((uint32_t)N, M, weighted, gs[0]->device, &u));
    pk->g = u;
    hipStream_t s = u->stream;
    Csr& c = u->out;
    c.n = (uint32_t)N;
    c.m = M;
    if (old && old->g && old->g->device == u->device) {
        eeg_graph* o = old->g;
        (void)hipStreamSynchronize(o->stream);
        carry(o->out.row, c.row, (N + 1) * 8);
        carry(o->out.col, c.col, M * 4);
        if (weighted) carry(o->out.w, c.w, M * 4);
        carry(o->perm, u->perm, N * 4);
        carry(o->inv, u->inv, N * 4);
        for (int i = 0; i < 4; ++i) {
            carry(o->tout[i].vlist, u->tout[i].vlist, N * 4);
            carry(o->tout[i].vscan, u->tout[i].vscan, N * 4);
            carry(o->tout[i].vnc, u->tout[i].vnc, N * 4);
        }
        carry(o->work.lab, u->work.lab, N * 4);
        carry(o->work.out, u->work.out, N * 4);
        for (int i = 0; i < 2; ++i) {
            carry(o->work.q[i], u->work.q[i], N * 4);
            carry(o->work.s[i], u->work.s[i], N * 4);
        }
        carry(o->work.mark, u->work.mark, N);
        carry(old->table, pk->table, k * sizeof(PackMember));
    }
    old.reset();
    EEG_TRY(c.row.alloc((N + 1) * 8));
    EEG_TRY(c.col.alloc(M * 4 + 4));
    if (weighted) EEG_TRY(c.w.alloc(M * 4 + 4));
    EEG_TRY(u->perm.alloc(N * 4 + 4));
    EEG_TRY(u->inv.alloc(N * 4 + 4));
    EEG_TRY(pk->seeds.alloc((size_t)k * 4 + 4));
    const size_t mbytes = k * sizeof(PackMember);
    EEG_TRY(pk->table.alloc(mbytes + chunks.size() * sizeof(PackChunk)));
    uint8_t* tab = pk->table.as<uint8_t>();
    EEG_HIP(hipMemcpyAsync(tab, mem.data(), mbytes, hipMemcpyHostToDevice, s));
    if (!chunks.empty())
        EEG_HIP(hipMemcpyAsync(tab + mbytes, chunks.data(), chunks.size() * sizeof(PackChunk), hipMemcpyHostToDevice, s));
    // the members' streams may still be writing their tables: wait for them first
    for (uint32_t i = 0; i < k; ++i) EEG_HIP(hipStreamSynchronize(gs[i]->stream));
    if (!chunks.empty()) {
        k_pack<<<(unsigned)chunks.size(), WG, 0, s>>>(reinterpret_cast<const PackChunk*>(tab + mbytes),
                                                      reinterpret_cast<const PackMember*>(tab), c.row.as<uint64_t>(),
                                                      c.col.as<uint32_t>(), weighted ? c.w.as<uint32_t>() : nullptr,
                                                      u->perm.as<uint32_t>(), u->inv.as<uint32_t>());
        EEG_HIP(hipGetLastError());
    }
    for (uint32_t i = 0; i < k; ++i) {
        if (i == 0 || gs[i]->max_deg > u->max_deg) {  // lowest id among the maxima
            u->max_deg = gs[i]->max_deg;
            u->argmax_deg = gs[i]->argmax_deg + pk->voff[i];
        }
        u->nonzero_out += gs[i]->nonzero_out;
    }
    if (N == 0) EEG_HIP(hipMemsetAsync(c.row.p, 0, 8, s));
    c.built = true;
    EEG_HIP(hipStreamSynchronize(s));
    return EEG_OK;
}

__global__ void k_unoffset(uint32_t* __restrict__ lab, uint64_t cnt, uint32_t off) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < cnt;
         i += (uint64_t)gridDim.x * blockDim.x)
        lab[i] -= off;
}

}  // namespace
}  // namespace eeg

using namespace eeg;

extern "C" eeg_status eeg_run_packed(eeg_graph* const* graphs, uint32_t ngraphs, uint32_t algo,
                                     const uint32_t* sources, const eeg_opts* opts,
                                     void* const* labels_out, eeg_stats* stats) {
    clear_error();
    if (!graphs || ngraphs == 0) return fail(EEG_ERR_INVALID_ARG, "no graphs");
    if (algo > EEG_PPR) return fail(EEG_ERR_INVALID_ARG, "unknown algorithm %u", algo);
    if (algo == EEG_PR || algo == EEG_PPR)
        return fail(EEG_ERR_UNSUPPORTED, "packed runs support BFS, SSSP, SSWP and CC");
    const bool sourced = algo != EEG_CC;
    if (sourced && !sources) return fail(EEG_ERR_INVALID_ARG, "null sources");
    for (uint32_t i = 0; i < ngraphs; ++i) {
        if (!graphs[i]) return fail(EEG_ERR_INVALID_ARG, "graph %u is null", i);
        if (sourced && sources[i] >= graphs[i]->n)
            return fail(EEG_ERR_INVALID_ARG, "source %u of graph %u out of range (n = %u)", sources[i], i,
                        graphs[i]->n);
    }
    eeg_opts o;
    memset(&o, 0, sizeof(o));
    if (opts) o = *opts;
    eeg_stats local;
    eeg_stats* st = stats ? stats : &local;
    memset(st, 0, sizeof(*st));
    const auto t0 = std::chrono::steady_clock::now();

    std::lock_guard<std::mutex> lk(g_pack_mu);
    DeviceGuard dg;
    EEG_TRY(select_device(graphs[0]->device));
    std::vector<uint64_t> key(ngraphs);
    for (uint32_t i = 0; i < ngraphs; ++i) key[i] = graphs[i]->serial;
    if (!g_pack || g_pack->serials != key) {
        std::unique_ptr<Packed> old(g_pack);
        g_pack = new (std::nothrow) Packed();
        if (!g_pack) return fail(EEG_ERR_OOM, "host allocation failed");
        eeg_status s = build_union(graphs, ngraphs, g_pack, std::move(old));
        if (s == EEG_ERR_OOM) {  // memory taken over may be larger than needed: once more without
            delete g_pack;
            g_pack = new (std::nothrow) Packed();
            if (!g_pack) return fail(EEG_ERR_OOM, "host allocation failed");
            s = build_union(graphs, ngraphs, g_pack, nullptr);
        }
        if (s != EEG_OK) {
            delete g_pack;
            g_pack = nullptr;
            return s;
        }
        g_pack->serials = key;
    }
    Packed& pk = *g_pack;
    eeg_graph* u = pk.g;
    std::lock_guard<std::mutex> lu(u->mu);
    hipStream_t s = u->stream;

    double e0 = 0, e1 = 0;
    const bool energy = o.energy && eeg_energy_read(u->device, &e0, nullptr) == EEG_OK;
    eeg_status rc;
    if (sourced) {
        std::vector<uint32_t> seeds(ngraphs);
        for (uint32_t i = 0; i < ngraphs; ++i) seeds[i] = graphs[i]->h_perm[sources[i]] + pk.voff[i];
        EEG_HIP(hipMemcpyAsync(pk.seeds.p, seeds.data(), (size_t)ngraphs * 4, hipMemcpyHostToDevice, s));
        rc = run_traversal(u, algo, 0, o, st, pk.seeds.as<uint32_t>(), ngraphs);
    } else {
        rc = run_traversal(u, algo, 0, o, st);
    }
    if (energy && eeg_energy_read(u->device, &e1, nullptr) == EEG_OK) st->energy_j = (e1 - e0) * 1e-6;
    if (rc != EEG_OK && rc != EEG_ERR_NOT_CONVERGED) return rc;
    const eeg_status keep = rc;
    if (labels_out && u->n) {
        EEG_TRY(u->work.out.alloc((size_t)u->n * 4 + 4));
        EEG_TRY(unpermute(u, u->work.lab.p, u->work.out.p, s, 0, u->n));
        uint32_t* outd = u->work.out.as<uint32_t>();
        for (uint32_t i = 0; i < ngraphs; ++i) {
            const uint32_t ni = pk.voff[i + 1] - pk.voff[i];
            if (!ni || !labels_out[i] || algo != EEG_CC || !pk.voff[i]) continue;
            k_unoffset<<<grid_pk(ni), WG, 0, s>>>(outd + pk.voff[i], ni, pk.voff[i]);
            EEG_HIP(hipGetLastError());
        }
        const size_t bytes = (size_t)u->n * 4;
        LentRing lent(u->device, bytes >= HOST_COPY_FROM);
        if (lent.r) {
            // the union's labels in slots, each cut at the graphs' bounds
            constexpr uint32_t words = HOST_SLOT_BYTES / 4;
            const uint32_t N = u->n, chunks = (uint32_t)(((uint64_t)N + words - 1) / words);
            EEG_TRY(stage_to_host(
                *lent.r, s, chunks, host_copy_threads(bytes), true,
                [&](uint32_t c, uint32_t count, void* slot) -> eeg_status {
                    EEG_HIP(hipMemcpyAsync(slot, outd + (size_t)c * words,
                                           (size_t)std::min<uint64_t>((uint64_t)count * words, N - c * words) * 4,
                                           hipMemcpyDeviceToHost, s));
                    return EEG_OK;
                },
                [&](uint32_t c, const void* slot, unsigned, unsigned) {
                    const uint32_t b = c * words, e = b + std::min(words, N - b);
                    uint32_t i = (uint32_t)(std::upper_bound(pk.voff.begin(), pk.voff.end(), b) - pk.voff.begin()) - 1;
                    for (; i < ngraphs && pk.voff[i] < e; ++i) {
                        const uint32_t lo = std::max(b, pk.voff[i]), hi = std::min(e, pk.voff[i + 1]);
                        if (lo < hi && labels_out[i])
                            memcpy((uint32_t*)labels_out[i] + (lo - pk.voff[i]), (const uint32_t*)slot + (lo - b),
                                   (size_t)(hi - lo) * 4);
                    }
                }));
        } else {
            for (uint32_t i = 0; i < ngraphs; ++i) {
                const uint32_t ni = pk.voff[i + 1] - pk.voff[i];
                if (!ni || !labels_out[i]) continue;
                EEG_HIP(hipMemcpyAsync(labels_out[i], outd + pk.voff[i], (size_t)ni * 4, hipMemcpyDeviceToHost, s));
            }
            EEG_HIP(hipStreamSynchronize(s));
        }
    }
    st->ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (keep != EEG_OK) return fail(keep, "no fixpoint within max_iters");
    return EEG_OK;
}
