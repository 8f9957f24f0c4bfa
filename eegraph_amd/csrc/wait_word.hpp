// Waiting on the host for a word that a kernel writes to pinned memory.  Host code only.
#pragma once

#include <cstdint>

namespace eeg {

enum class Queue { BUSY, DRAINED, FAILED };  // state of the stream that the kernel is queued on

// Returns once *word is other than `not_yet`, or false if the stream has drained or failed without
// it.  query() tells the stream's state; it costs a call to the runtime, so it is asked now and then.
template <class Query>
bool wait_word(const volatile uint64_t* word, uint64_t not_yet, Query query) {
    for (uint32_t spins = 1; *word == not_yet; ++spins) {
        // (what a drained stream wrote came before its end: one more look decides)
        if ((spins & 0x3fff) == 0 && query() != Queue::BUSY) return *word != not_yet;
        __builtin_ia32_pause();
    }
    return true;
}

}  // namespace eeg
