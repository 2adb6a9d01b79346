"""Scratch memory that grows (internal.hpp, grow) when an allocation fails, on the host with an
allocator that refuses: the call reports it, and a later, smaller one allocates again instead of
taking the size that had been there before.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "internal.hpp"
static size_t most = 1 << 20;
static int live = 0;
extern "C" hipError_t hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (n > most) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    ++live;
    return hipSuccess;
}
extern "C" hipError_t hipFree(void* p) {
    std::free(p);
    --live;
    return hipSuccess;
}
int main() {
    double* p = nullptr;
    long cap = 0;
    hpq::grow(p, cap, 1000);
    if (!p || cap != 1000 || live != 1) return 1;
    double* const first = p;
    hpq::grow(p, cap, 10);
    if (p != first || cap != 1000) return 2;
    bool thrown = false;
    try {
        hpq::grow(p, cap, 1 << 20);
    } catch (const hpq::HipError&) {
        thrown = true;
    }
    if (!thrown || live != 0) return 3;
    hpq::grow(p, cap, 500);
    return p && cap == 500 && live == 1 ? 0 : 4;
}
"""


def test_grow_after_a_failed_allocation(tmp_path):
    src, exe = tmp_path / "scratch.hip", tmp_path / "scratch"
    src.write_text(PROGRAM)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.run([hipcc, "-O1", "-std=c++17", "-x", "hip", "--offload-host-only",
                    "-I", os.path.join(ROOT, "hipace2_amd", "csrc"), "-o", str(exe), str(src)], check=True,
                   capture_output=True, timeout=300)
    assert subprocess.run([str(exe)], timeout=60).returncode == 0
