// Large answers on their way to a caller's host memory, and large edge lists on their way from it.
//
// What bounds it: hipMemcpy into pageable memory moves 256 MiB in 16 ms where the pages exist and in
// 26 ms where the caller has just allocated them (one thread copies and takes the page faults); PCIe
// takes 5 ms of that.  So a kernel writes an answer in slots of pinned memory, in the order and layout
// the caller wants, and several threads copy finished slots out while the next ones are written.
// Towards the device the threads fill the slots (192 MiB of edges: 8.2 ms as plain copies).
#pragma once

#include <algorithm>
#include <atomic>
#include <exception>
#include <thread>
#include <vector>

#include "engine.hpp"

namespace eeg {

// Slots of pinned memory and an event for each.  Rings are lent by a pool that keeps at most
// HOST_RINGS_KEPT of them between calls (pinning 32 MiB takes milliseconds).
constexpr uint32_t HOST_SLOTS = 16;
constexpr size_t HOST_SLOT_BYTES = (size_t)2 << 20;
constexpr size_t HOST_RINGS_KEPT = 2;
// Slots, neighbours in the ring, that one launch or copy covers at most: each costs about 13 us
// beyond its transfer (256 MiB in 128 launches 6.8 ms, in 32 5.5).  Threads take single slots.
constexpr uint32_t HOST_GROUP = 4;
constexpr unsigned HOST_THREADS = 8;
struct HostRing {
    int device = 0;
    uint8_t* base = nullptr;
    hipEvent_t ev[HOST_SLOTS] = {};
    void* slot(uint32_t i) const { return base + (size_t)(i % HOST_SLOTS) * HOST_SLOT_BYTES; }
    ~HostRing();
};
// A ring for the current device, or null (no memory: the caller takes the plain copy).
HostRing* take_host_ring(int device);
void give_host_ring(HostRing* r);

// From 8 MiB on: a plain copy of 4 MiB takes 0.25 .. 0.4 ms, of which threads would save what
// starting them costs.
constexpr uint64_t HOST_COPY_FROM = (uint64_t)8 << 20;
inline unsigned host_copy_threads(uint64_t bytes) {
    const unsigned hw = std::thread::hardware_concurrency();
    const unsigned most = std::max(1u, std::min(HOST_THREADS, hw / 2));
    return (unsigned)std::min<uint64_t>(most, std::max<uint64_t>(1, bytes / (2 * HOST_SLOT_BYTES)));
}

// Chunks that go together from `first` on, not past the ring's end.  Few chunks make small groups,
// so that the two sides still overlap.
inline uint32_t host_group(uint32_t first, uint32_t chunks) {
    const uint32_t most = std::max(1u, std::min(HOST_GROUP, chunks / 8));
    return std::min(std::min(most, chunks - first), HOST_SLOTS - first % HOST_SLOTS);
}

// Runs chunks 0 .. chunks-1 through the ring: produce(i, count, slot) queues on stream s what fills
// the slots from `slot` on with chunks i .. i + count - 1, take(i, slot, w, nw) copies share w of nw of it to where it belongs, on one of
// `threads` threads.  `whole`: every chunk goes to one thread (nw = 1) rather than a share of it to
// each; what a thread touches first should be pages that no other thread touches.
template <class Produce, class Take>
eeg_status stage_to_host(HostRing& ring, hipStream_t s, uint32_t chunks, unsigned threads, bool whole,
                         Produce produce, Take take) {
    std::atomic<uint32_t> ready{0}, left[HOST_SLOTS];
    std::atomic<unsigned> team{0};  // threads that share the work, once all have started
    std::atomic<bool> stop{false};
    auto work = [&](unsigned w) {
        unsigned nw;
        while (!(nw = team.load(std::memory_order_acquire)))
            if (stop.load(std::memory_order_relaxed)) return;
            else __builtin_ia32_pause();
        for (uint32_t i = 0; i < chunks; ++i) {
            if (whole && i % nw != w) continue;
            for (uint32_t spins = 1; ready.load(std::memory_order_acquire) <= i; ++spins) {
                if (stop.load(std::memory_order_relaxed)) return;
                if (spins % 64) __builtin_ia32_pause();
                else std::this_thread::yield();
            }
            if (whole) take(i, ring.slot(i), 0u, 1u);
            else take(i, ring.slot(i), w, nw);
            left[i % HOST_SLOTS].fetch_sub(1, std::memory_order_release);
        }
    };
    std::vector<std::thread> pool;
    unsigned started = 0;
    try {
        pool.reserve(threads);
        for (; started < threads; ++started) pool.emplace_back(work, started);
    } catch (const std::exception&) {  // fewer threads, or none, do as well
    }
    const uint32_t shares = whole ? 1u : std::max(1u, started);
    for (auto& l : left) l.store(shares, std::memory_order_relaxed);
    team.store(std::max(1u, started), std::memory_order_release);
    eeg_status rc = EEG_OK;
    uint32_t queued = 0, seen = 0, freed = 0;
    while (rc == EEG_OK && freed < chunks) {
        while (queued < chunks) {
            const uint32_t count = host_group(queued, chunks);
            if (queued + count > freed + HOST_SLOTS) break;
            rc = produce(queued, count, ring.slot(queued));
            queued += count;
            // the event of a group is that of its last slot
            if (rc == EEG_OK && hipEventRecord(ring.ev[(queued - 1) % HOST_SLOTS], s) != hipSuccess)
                rc = fail(EEG_ERR_DEVICE, "hipEventRecord failed");
            if (rc != EEG_OK) break;
        }
        if (rc != EEG_OK) break;
        if (seen < queued) {
            const uint32_t count = host_group(seen, chunks);
            const hipError_t e = hipEventQuery(ring.ev[(seen + count - 1) % HOST_SLOTS]);
            if (e == hipSuccess) {
                for (uint32_t i = seen; !started && i < seen + count; ++i) {
                    take(i, ring.slot(i), 0u, 1u);
                    left[i % HOST_SLOTS].store(0, std::memory_order_relaxed);
                }
                seen += count;
                ready.store(seen, std::memory_order_release);
            } else if (e != hipErrorNotReady) {
                rc = fail(EEG_ERR_DEVICE, "copy to the host failed: %s", hipGetErrorString(e));
                break;
            } else {
                (void)hipGetLastError();  // "not ready" is no error of the next launch
            }
        }
        while (freed < seen && left[freed % HOST_SLOTS].load(std::memory_order_acquire) == 0) {
            left[freed % HOST_SLOTS].store(shares, std::memory_order_relaxed);
            ++freed;
        }
        __builtin_ia32_pause();
    }
    if (rc != EEG_OK) {
        stop.store(true);
        (void)hipStreamSynchronize(s);  // what is queued writes to the slots
    }
    for (auto& t : pool) t.join();
    return rc;
}

// The other way: fill(i, slot) writes chunk i into its slot on one of `threads` threads, consume(i,
// count, slot) queues on stream s, in order, what reads the slots from `slot` on, which hold chunks i
// .. i + count - 1.  Returns when all of it has been read.
template <class Fill, class Consume>
eeg_status stage_to_device(HostRing& ring, hipStream_t s, uint32_t chunks, unsigned threads, Fill fill,
                           Consume consume) {
    std::atomic<uint32_t> freed{0}, filled[HOST_SLOTS];  // filled: one past the chunk in the slot
    std::atomic<unsigned> team{0};
    std::atomic<bool> stop{false};
    for (auto& f : filled) f.store(0, std::memory_order_relaxed);
    auto work = [&](unsigned w) {
        unsigned nw;
        while (!(nw = team.load(std::memory_order_acquire))) __builtin_ia32_pause();
        for (uint32_t i = w; i < chunks; i += nw) {
            for (uint32_t spins = 1; i >= freed.load(std::memory_order_acquire) + HOST_SLOTS; ++spins) {
                if (stop.load(std::memory_order_relaxed)) return;
                if (spins % 64) __builtin_ia32_pause();
                else std::this_thread::yield();
            }
            fill(i, ring.slot(i));
            filled[i % HOST_SLOTS].store(i + 1, std::memory_order_release);
        }
    };
    std::vector<std::thread> pool;
    unsigned started = 0;
    try {
        pool.reserve(threads);
        for (; started < threads; ++started) pool.emplace_back(work, started);
    } catch (const std::exception&) {  // fewer threads, or none, do as well
    }
    team.store(std::max(1u, started), std::memory_order_release);
    eeg_status rc = EEG_OK;
    uint32_t queued = 0, done = 0;
    uint32_t full = 0;  // chunks seen filled, in order
    while (rc == EEG_OK && done < chunks) {
        if (!started && full < chunks && full < done + HOST_SLOTS) {
            fill(full, ring.slot(full));
            filled[full % HOST_SLOTS].store(full + 1, std::memory_order_relaxed);
        }
        while (full < chunks && filled[full % HOST_SLOTS].load(std::memory_order_acquire) == full + 1) ++full;
        if (queued < chunks && full >= queued + host_group(queued, chunks)) {
            const uint32_t count = host_group(queued, chunks);
            rc = consume(queued, count, ring.slot(queued));
            queued += count;
            if (rc == EEG_OK && hipEventRecord(ring.ev[(queued - 1) % HOST_SLOTS], s) != hipSuccess)
                rc = fail(EEG_ERR_DEVICE, "hipEventRecord failed");
            if (rc != EEG_OK) break;
        }
        if (done < queued) {
            const uint32_t count = host_group(done, chunks);
            const hipError_t e = hipEventQuery(ring.ev[(done + count - 1) % HOST_SLOTS]);
            if (e == hipSuccess) {
                done += count;
                freed.store(done, std::memory_order_release);
            } else if (e != hipErrorNotReady) {
                rc = fail(EEG_ERR_DEVICE, "copy to the device failed: %s", hipGetErrorString(e));
                break;
            } else {
                (void)hipGetLastError();  // "not ready" is no error of the next launch
            }
        }
        __builtin_ia32_pause();
    }
    if (rc != EEG_OK) {
        stop.store(true);
        (void)hipStreamSynchronize(s);  // what is queued reads the slots
    }
    for (auto& t : pool) t.join();
    return rc;
}

// The ring of one call; given back when it ends.
struct LentRing {
    HostRing* r;
    explicit LentRing(int device, bool wanted) : r(wanted ? take_host_ring(device) : nullptr) {}
    ~LentRing() {
        if (r) give_host_ring(r);
    }
    LentRing(const LentRing&) = delete;
    LentRing& operator=(const LentRing&) = delete;
};

}  // namespace eeg
