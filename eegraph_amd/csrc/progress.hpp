// Progress of a traversal, reported by its kernels as its iterations start: the host queues a few
// iterations ahead of it and stops with the one that finds nothing to do.  Shared by the
// single-query traversals (relax.hip) and the batched passes (batch.hip).
#pragma once

#include "engine.hpp"

namespace eeg {

enum RunState : uint32_t { RUN_GOING = 0, RUN_DONE = 1, RUN_ERROR = 2 };

// Written to pinned memory by one thread.  The words are independent (the host waits for each on
// its own), so relaxed stores do.
__device__ __forceinline__ void publish(RunStatus* st, const Ctl* ctl, uint32_t it, uint32_t state) {
    if (!st) return;
    const unsigned long long now = (unsigned long long)wall_clock64();
    if (it == 1) __hip_atomic_store(&st->t0, now, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (state == RUN_DONE) __hip_atomic_store(&st->t1, now, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (ctl->err) state = RUN_ERROR;
    __hip_atomic_store(&st->word, ((unsigned long long)it << 8) | state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Iterations queued beyond the one that the device is known to have started: enough that it never
// waits for the host (an iteration takes 9 us or more, seeing it start and queueing the next about
// 8), and what is left to run dry after the last one is short.
constexpr uint32_t RUN_AHEAD = 2;

// Clears the status before a run.  (Nothing of an earlier run writes it any more: a run ends when its
// last status is seen, or with its stream synchronised.)
inline void reset_status(RunStatus* status) {
    volatile RunStatus* vs = status;
    vs->word = 0;
    vs->t0 = 0;
    vs->t1 = 0;
}

// Launches iterations *it, *it + 1, .. (launch(i) queues iteration i on stream s), at most `limit` of
// them, until the status says RUN_DONE or RUN_ERROR or the last one has run without; *state is what
// was seen then.
template <class Launch>
eeg_status run_ahead(hipStream_t s, RunStatus* status, uint64_t limit, uint32_t* it, uint32_t* state, Launch launch) {
    volatile RunStatus* vs = status;
    uint64_t started = 0;
    for (uint32_t spins = 1;; ++spins) {
        while (*it <= limit && *it <= started + RUN_AHEAD) EEG_TRY(launch((*it)++));
        const unsigned long long word = vs->word;
        *state = (uint32_t)(word & 0xff);
        if (*state != RUN_GOING) return EEG_OK;
        if (word >> 8 != started) {
            started = word >> 8;
            spins = 0;
            continue;
        }
        if ((spins & 0x3fff) == 0) {  // a device error ends the wait; so does the last iteration
            const hipError_t e = hipStreamQuery(s);
            if (e == hipSuccess && *it > limit && vs->word == word) return EEG_OK;
            if (e != hipSuccess && e != hipErrorNotReady)
                return fail(EEG_ERR_DEVICE, "traversal failed: %s", hipGetErrorString(e));
            (void)hipGetLastError();  // "not ready" is no error of the next launch
        }
        __builtin_ia32_pause();
    }
}

// Ticks of the device clock (wall_clock64) per millisecond.
inline double clock_khz(int device) {
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device) != hipSuccess || khz <= 0) khz = 100000;
    return (double)khz;
}

// Device time of a run, from the start of its first iteration to the one that found nothing to do, or
// to the end of the last one admitted.
inline double run_ms(const RunStatus* status, int device) {
    const volatile RunStatus* vs = status;
    while (!vs->t1) __builtin_ia32_pause();
    return (double)(vs->t1 - vs->t0) / clock_khz(device);
}

}  // namespace eeg
