"""Cutting host edge lists into slots (eegraph_amd/csrc/upload_chunks.hpp): every byte of every array
arrives once and nothing is written beside an array, also where the arrays lie next to each other or
exactly a slot behind another's last, partial chunk.  Compiled for the host with the ROCm clang."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANG = "/opt/rocm/llvm/bin/clang++"

HARNESS = r"""
#include <cstdio>
#include <cstring>
#include <vector>
#include "upload_chunks.hpp"
using namespace eeg;

// Arrays of the given bytes at the given places of one "device" memory, uploaded in groups.
static bool check(const std::vector<size_t>& bytes, const std::vector<size_t>& at, size_t slot, uint32_t group) {
    std::vector<uint8_t> dev(4096, 0), want(4096, 0);
    std::vector<std::vector<uint8_t>> host;
    std::vector<Upload> parts;
    for (size_t p = 0; p < bytes.size(); ++p) {
        host.emplace_back(bytes[p]);
        for (size_t i = 0; i < bytes[p]; ++i) want[at[p] + i] = host[p][i] = (uint8_t)(1 + (31 * p + i) % 250);
    }
    for (size_t p = 0; p < bytes.size(); ++p) parts.push_back(Upload{dev.data() + at[p], host[p].data(), bytes[p]});
    const UploadChunks chunks{parts.data(), parts.size(), slot};
    for (uint32_t i = 0; i < chunks.count(); i += group) {
        const uint32_t n = std::min(group, chunks.count() - i);
        std::vector<uint8_t> slots(n * slot, 0xee);
        for (uint32_t k = 0; k < n; ++k) {
            const Upload c = chunks[i + k];
            if (!c.bytes || c.bytes > slot) return false;
            memcpy(slots.data() + k * slot, c.src, c.bytes);
        }
        const bool ok = chunks.runs(i, n, [&](void* dst, size_t off, size_t b) {
            bool inside = false;  // one array: they are allocations of their own
            for (const Upload& u : parts)
                inside |= (uint8_t*)dst >= (uint8_t*)u.dst && (uint8_t*)dst + b <= (uint8_t*)u.dst + u.bytes;
            if (off + b > slots.size() || !inside) return false;
            memcpy(dst, slots.data() + off, b);
            return true;
        });
        if (!ok) return false;
    }
    return dev == want;
}

int main() {
    int bad = 0;
    auto expect = [&](bool ok, const char* what, size_t a, uint32_t g) {
        if (!ok && ++bad) printf("wrong: %s, %zu bytes, groups of %u\n", what, a, g);
    };
    const size_t slot = 16;
    for (uint32_t g = 1; g <= 4; ++g)
        for (size_t a = 0; a <= 5 * slot; ++a) {
            const size_t full = a / slot * slot;
            expect(check({a, a, a}, {0, 1000, 2000}, slot, g), "apart", a, g);
            expect(check({a, a, a}, {0, a, 2 * a}, slot, g), "side by side", a, g);
            // the second array a slot behind the start of the first one's last chunk
            expect(check({a, a, a}, {0, full + slot, 2 * (full + slot)}, slot, g), "a slot apart", a, g);
            expect(check({a, 0, a}, {0, full + slot, full + slot}, slot, g), "an empty array between", a, g);
            expect(check({a, a}, {2000, 0}, slot, g), "the other way round", a, g);
        }
    printf("wrong %d\n", bad);
    return bad != 0;
}
"""


@pytest.mark.skipif(not os.path.exists(CLANG), reason="needs the ROCm clang")
def test_chunks_go_to_their_own_array(tmp_path):
    src = tmp_path / "upload_check.cpp"
    src.write_text(HARNESS)
    exe = tmp_path / "upload_check"
    subprocess.run([CLANG, "-O1", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "eegraph_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "wrong 0" in r.stdout
