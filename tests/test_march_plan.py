"""The chunk of the marched red-black launches (fit_march, a host function that
runs for every launch): the one an exhaustive search finds, in time that does
not grow with the grid's depth."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = "/opt/rocm/llvm/bin/clang++"
SOURCE = r"""
#include <chrono>
#include <cstdio>
#include "smoke_internal.h"
using smk::MarchChunk;
static MarchChunk all(long long columns, int planes, int fill)
{
    MarchChunk best{planes, -1};
    for (int chunks = 1; chunks <= (planes + 1) / 2; ++chunks) {
        const int zc = (planes + chunks - 1) / chunks;
        const long long blocks = columns * ((planes + zc - 1) / zc);
        const long long steps = (blocks + smk::kCUs - 1) / smk::kCUs * (zc + fill);
        if (best.steps < 0 || steps < best.steps) best = {zc, steps};
    }
    return best;
}
int main()
{
    for (int fill : {8, 12, 15, 18})
        for (long long columns : {1, 2, 3, 7, 16, 30, 63, 64, 100, 255, 256, 257, 300, 1000, 5000})
            for (int planes = 1; planes < 3000; planes += planes < 200 ? 1 : 41) {
                const MarchChunk a = all(columns, planes, fill), b = smk::fit_march(columns, planes, fill);
                if (a.zc != b.zc || a.steps != b.steps) {
                    printf("%lld columns, %d planes, fill %d: %d %lld, exhaustive %d %lld\n", columns,
                           planes, fill, b.zc, b.steps, a.zc, a.steps);
                    return 1;
                }
            }
    const auto t0 = std::chrono::steady_clock::now();
    long long sum = 0;
    for (int k = 0; k < 1000; ++k) sum += smk::fit_march(1 + k % 3, 8000000 - k, 12).steps;
    const double s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    printf("%.6f s for 1000 deep grids (%lld)\n", s, sum);
    return s < 2.0 ? 0 : 2;  // 12 s with every chunk tried
}
"""


@pytest.mark.skipif(not os.path.exists(CXX), reason="host clang++ is not available")
def test_fitted_march_chunks(tmp_path):
    src, exe = tmp_path / "march.cpp", tmp_path / "march"
    src.write_text(SOURCE)
    r = subprocess.run([CXX, "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "smoke-simulation_amd", "csrc"), str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
