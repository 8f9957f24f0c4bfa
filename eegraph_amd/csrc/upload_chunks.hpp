// Host arrays on their way to the device through pinned slots (hostcopy.hpp): how they are cut into
// chunks of a slot each, and which neighbouring chunks go in one copy.  Host code only.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace eeg {

// A host array (or a piece of one) and the device memory it goes to.
struct Upload {
    void* dst;
    const void* src;
    size_t bytes;
};

// Chunks of `slot` bytes of the arrays in turn; the last chunk of an array may be shorter, and
// arrays of no bytes have none.
struct UploadChunks {
    const Upload* parts;
    size_t nparts;
    size_t slot;

    uint32_t of(size_t p) const { return (uint32_t)((parts[p].bytes + slot - 1) / slot); }
    uint32_t count() const {
        uint32_t n = 0;
        for (size_t p = 0; p < nparts; ++p) n += of(p);
        return n;
    }
    // Chunk i < count(); *part: the array it is cut from.
    Upload chunk(uint32_t i, size_t* part) const {
        size_t p = 0;
        for (; i >= of(p); ++p) i -= of(p);
        *part = p;
        const size_t o = (size_t)i * slot;
        return Upload{(uint8_t*)parts[p].dst + o, (const uint8_t*)parts[p].src + o, std::min(slot, parts[p].bytes - o)};
    }
    Upload operator[](uint32_t i) const {
        size_t p;
        return chunk(i, &p);
    }
    // Chunks first .. first + count - 1, which lie slot by slot in pinned memory, as one copy per
    // array: copy(dst, offset in the pinned memory, bytes) for each, until one fails.  Arrays are
    // allocations of their own, so a copy never goes on into the next one, wherever that lies (all
    // but an array's last chunk fill their slots: an array's chunks follow each other on both sides).
    template <class Copy>
    bool runs(uint32_t first, uint32_t count, Copy copy) const {
        for (uint32_t k = 0; k < count;) {
            size_t array, next;
            const Upload c = chunk(first + k, &array);
            size_t bytes = c.bytes;
            uint32_t e = k + 1;
            for (; e < count; ++e) {
                const Upload x = chunk(first + e, &next);
                if (next != array) break;
                bytes += x.bytes;
            }
            if (!copy(c.dst, (size_t)k * slot, bytes)) return false;
            k = e;
        }
        return true;
    }
};

}  // namespace eeg
