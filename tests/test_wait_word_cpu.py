"""The host's wait for a word in pinned memory (eegraph_amd/csrc/wait_word.hpp) ends with the word, with
a failed stream and with one that has drained without writing it; a word that came just before the
stream drained counts.  A thread stands in for the kernel; compiled for the host with the ROCm clang."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANG = "/opt/rocm/llvm/bin/clang++"

HARNESS = r"""
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include "wait_word.hpp"
using namespace eeg;
int main() {
    const uint64_t none = ~0ull;
    volatile uint64_t word = none;
    int bad = 0;
    auto expect = [&](bool ok, const char* what) { if (!ok) { ++bad; printf("wrong: %s\n", what); } };
    std::thread kernel([&] { std::this_thread::sleep_for(std::chrono::milliseconds(20)); word = 7; });
    expect(wait_word(&word, none, [] { return Queue::BUSY; }), "a word from a busy stream");
    kernel.join();
    expect(wait_word(&word, none, [] { return Queue::FAILED; }), "a word that is there already");
    word = none;
    expect(!wait_word(&word, none, [] { return Queue::FAILED; }), "a failed stream");
    expect(!wait_word(&word, none, [] { return Queue::DRAINED; }), "a drained stream without the word");
    int asked = 0;
    expect(wait_word(&word, none, [&] { if (++asked == 3) { word = 9; return Queue::DRAINED; } return Queue::BUSY; }),
           "a word written just before the stream drained");
    printf("wrong %d\n", bad);
    return bad != 0;
}
"""


@pytest.mark.skipif(not os.path.exists(CLANG), reason="needs the ROCm clang")
def test_every_wait_ends(tmp_path):
    src = tmp_path / "wait_check.cpp"
    src.write_text(HARNESS)
    exe = tmp_path / "wait_check"
    subprocess.run([CLANG, "-O2", "-std=c++17", "-Wall", "-pthread", "-I", os.path.join(ROOT, "eegraph_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
