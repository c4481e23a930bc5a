"""The threads that copy a large table into pinned chunks (csrc/copy_threads.hpp), as a host
program of its own: no GPU is needed."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <stdexcept>

#include "copy_threads.hpp"

static long g_left = -1;   // allocations of the calling thread until one fails; negative: none does
static thread_local bool t_main = false;
void* operator new(size_t n) {
    if (t_main && g_left >= 0 && g_left-- == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

int main() {
    t_main = true;
    const unsigned kWant = 4, kChunks = 9, kFeatures = 11;
    int whole = 0, refused = 0;
    for (long fail = -1; fail < 12; ++fail) {   // none, the chunk counters, the pool, each thread
        for (int broken_off = 0; broken_off < 2; ++broken_off) {
            unsigned char seen[kChunks][kFeatures] = {};
            auto copy = [&](uint64_t c, uint32_t first, uint32_t step) {
                for (uint32_t f = first; f < kFeatures; f += step) ++seen[c][f];
            };
            g_left = fail;
            try {
                cbh::CopyThreads<decltype(copy)> threads(kWant, kChunks, 2, copy);
                g_left = -1;
                for (uint64_t c = 0; c < kChunks; ++c) {
                    threads.wait(c);
                    for (uint32_t f = 0; f < kFeatures; ++f)
                        if (seen[c][f] != 1) return std::printf("chunk %d feature %u: %d\n", (int)c, f, seen[c][f]), 1;
                    if (broken_off && c == 3) throw std::runtime_error("caller");
                    threads.open(c + 3);
                }
                ++whole;
            } catch (const std::bad_alloc&) {
                ++refused;
            } catch (const std::runtime_error&) {
            }
            g_left = -1;
        }
    }
    std::printf("%d whole, %d refused\n", whole, refused);
    return 0;
}
"""


WAITING = r"""
#include <chrono>
#include <cstdio>
#include <ctime>

#include "copy_threads.hpp"

static double cpu() {
    timespec t;
    clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t);
    return t.tv_sec + 1e-9 * t.tv_nsec;
}

int main() {
    std::atomic<int> copies{0};
    auto slow = [&](uint64_t c, uint32_t, uint32_t) {   // chunk 1: the caller waits for its threads
        if (c == 1) std::this_thread::sleep_for(std::chrono::milliseconds(400));
        ++copies;
    };
    const double t0 = cpu();
    {
        cbh::CopyThreads<decltype(slow)> threads(4, 3, 2, slow);
        threads.wait(0);
        threads.wait(1);
        std::this_thread::sleep_for(std::chrono::milliseconds(400));   // its threads wait for chunk 2
        threads.open(3);
        threads.wait(2);
    }
    std::printf("%d copies, %.3f\n", copies.load(), cpu() - t0);
    return 0;
}
"""


def _run(tmp_path, program):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(program)
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I",
                    os.path.join(ROOT, "catboost_rs_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    return r.stdout


def test_waiting_threads_sleep(tmp_path):
    """400 ms in which the caller waits for its threads and 400 ms in which they wait for it: threads
    that only gave way would run for 0.4 s of CPU time or more in each, sleeping ones for almost none."""
    copies, cpu = _run(tmp_path, WAITING).split(" copies, ")
    assert copies == "12" and float(cpu) < 0.2


def test_copy_threads_survive_failed_starts(tmp_path):
    """A thread that cannot be started (its allocation fails) costs neither the call nor the process:
    the table is copied once by those there, by the caller if there is none, and a caller that
    breaks off with an exception in the middle leaves no thread behind."""
    assert _run(tmp_path, PROGRAM) == "11 whole, 4 refused\n"
