"""The on-chip PCG loads the matrix a step ahead of its test whether the step exists: every shape and
mesh size keeps those loads inside the tables, and real steps at their own rows (host code of
mpflow_amd/csrc/chip.h and chip.hip, no GPU)."""
import os
import subprocess

from tests.conftest import ROOT

SOURCE = r"""
#include <cstdio>
#include "chip.h"
int main() {
    long long steps = 0, past = 0;
    for (int np = 256; np <= mpf::kChipMaxRows; np += 256)
        for (int width : {8, 16, 32})
            for (long long lanes : {1LL, 256LL, 512LL, 1024LL, 100000LL}) {
                const mpf::ChipShape c = mpf::chip_shape(np, width, lanes);
                const int nw = c.threads / 64;
                if (c.G < 1 || c.K < 1 || c.threads % 64 || c.threads * c.K < np) return 2;
                for (int w = 0; w < nw; ++w)
                    for (int k = 0; k < c.K; ++k, ++steps) {
                        const int at = (w + k * nw) * 64, first = w * 64 + mpf::chip_step(k, w, nw, np);
                        if (first < 0 || first + 64 > np) {
                            std::printf("rows %d, width %d, lanes %lld: step %d of wavefront %d at %d\n", np, width,
                                        lanes, k, w, first);
                            return 1;
                        }
                        if (at < np && first != at) return 3;
                        past += at >= np;
                    }
            }
    std::printf("%lld steps, %lld past the rows\n", steps, past);
    return past ? 0 : 4;
}
"""


def test_loads_ahead_stay_inside_the_tables(tmp_path):
    src, exe, lib = tmp_path / "rows.cpp", tmp_path / "rows", os.path.join(ROOT, "mpflow_amd")
    src.write_text(SOURCE)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(lib, "csrc"),
                    "-I" + os.path.join(rocm, "include"), str(src), "-o", str(exe), "-L" + lib, "-l:libmpflow_amd.so",
                    "-Wl,-rpath," + lib, "-Wl,-rpath," + os.path.join(rocm, "lib"), "-L" + os.path.join(rocm, "lib"),
                    "-lamdhip64"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
