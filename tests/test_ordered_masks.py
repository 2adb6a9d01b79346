"""The part of a particle's stencil that lies in a block of cells (ordered.hpp, stencil_bits), which
decides where the ordered depositions write, on the host: every position of a stencil of 1 to 6
cells around blocks of 1 to 16, the stencils beyond the block's last cell among them, which belong
to particles outside the plane.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "ordered.hpp"
int main() {
    int wrong = 0;
    for (int S = 1; S <= 6; ++S)
        for (int cells = 1; cells <= 16; ++cells)
            for (int x = -(S - 1); x <= 20; ++x) {   // the stencil's first cell, counted from the block's
                unsigned want = 0;
                for (int k = 0; k < S; ++k)
                    if (x + k >= 0 && x + k < cells) want |= 1u << k;
                const unsigned got = hpq::stencil_bits(-x, cells - x, S);
                if (got != want && ++wrong <= 5) std::printf("S %d cells %d x %d: %x, not %x\n", S, cells, x, got, want);
            }
    return wrong != 0;
}
"""


def test_stencil_bits(tmp_path):
    src, exe = tmp_path / "masks.hip", tmp_path / "masks"
    src.write_text(PROGRAM)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.run([hipcc, "-O1", "-std=c++17", "-x", "hip", "--offload-host-only",
                    "-I", os.path.join(ROOT, "hipace2_amd", "csrc"), "-o", str(exe), str(src)], check=True,
                   capture_output=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
