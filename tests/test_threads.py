"""Host threads of large network reads (mpflow_amd/csrc/threads.h): where a thread cannot be started --
its constructor throws std::system_error or std::bad_alloc -- the others do the work and all are
joined, whatever the number that could be started."""
import os
import subprocess

from tests.conftest import ROOT

SOURCE = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include "threads.h"
static long left = 1 << 30;                 // allocations until the next one fails, on this thread
static std::atomic<bool> armed{false};
void* operator new(std::size_t n) {
    if (armed && left-- <= 0) throw std::bad_alloc();
    return std::malloc(n);
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
int main() {
    for (int started = 0; started < 9; ++started) {
        std::atomic<int> next{0}, done{0};
        left = started;                     // the vector's memory, then one allocation per thread
        armed = true;
        mpf::on_threads(8, [&](int) {
            while (next.fetch_add(1) < 1000) done.fetch_add(1);
        });
        armed = false;
        if (done != 1000) return 1;
    }
    return 0;
}
"""


def test_threads_that_cannot_start_leave_their_work_to_the_others(tmp_path):
    src, exe = tmp_path / "threads.cpp", tmp_path / "threads"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-w", "-pthread", "-I" + os.path.join(ROOT, "mpflow_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
