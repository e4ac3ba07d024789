"""A caught allocation failure leaves nothing behind: the callers that go on without the memory (the
on-chip tables, the inverse blocks, split products) launch kernels next, and the check after a launch
reads the runtime's last error.  Host code of mpflow_amd/csrc/mpf_internal.h over a stand-in for the
runtime whose failed calls stay recorded until they are read, as HIP's do."""
import os
import subprocess

from tests.conftest import ROOT

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include "mpf_internal.h"
static hipError_t last = hipSuccess;
static bool full = true;
static hipError_t allocate(void** p, size_t n) {
    if (full) return last = hipErrorOutOfMemory;
    *p = std::malloc(n);
    return hipSuccess;
}
extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return allocate(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) { return allocate(p, n); }
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipGetLastError(void) { const hipError_t e = last; last = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
}
int main() {
    mpf::DBuf<double> b;
    for (int host = 0; host < 2; ++host) {
        bool caught = false;
        try {
            if (host) (void)mpf::pinned_alloc<int>(100);
            else b.alloc(100);
        } catch (const mpf::Error& e) {
            caught = e.code == MPF_ENOMEM;
        }
        if (!caught || b.p || b.n) return 1;
        MPF_HIP(hipGetLastError());          // as after the next launch
    }
    full = false;
    b.alloc(100);
    int* h = mpf::pinned_alloc<int>(100);
    if (!b.p || !h) return 2;
    (void)hipHostFree(h);
    return 0;
}
"""


def test_caught_allocation_failure_is_not_reported_by_the_next_launch(tmp_path):
    src, exe = tmp_path / "nomem.cpp", tmp_path / "nomem"
    src.write_text(SOURCE)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "mpflow_amd", "csrc"),
                    "-I" + os.path.join(rocm, "include"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
