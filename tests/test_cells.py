"""The cell a trilinear sample reads, for any float coordinate: its loads do not wait for the test that the point is
inside, so the index must lie in the model whatever the coordinate is (CPU: the function is the kernel's)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

SRC = r"""
#include <cmath>
#include <cstdio>
#include <cstdint>
#include "emc_internal.h"
#include "hip/geom.h"
int main()
{
    int bad = 0;
    for (int L : {4, 5, 64, 1024}) {
        const float hi = (float)(L - 2);
        auto want = [&](float u, int c) {
            if (emc::nearest_cell(u, L) == c) return;
            std::printf("L %d u %g: %d, not %d\n", L, (double)u, emc::nearest_cell(u, L), c);
            ++bad;
        };
        for (int k = 0; k < L - 1; ++k) {  // inside: the floor, and at the upper edge the last cell
            want((float)k, k);
            want(std::nextafterf((float)(k + 1), 0.0f), k);
        }
        want((float)(L - 1), L - 2);
        for (float u : {-0.0f, -1.0f, -2147483904.0f, -1e30f, -INFINITY, (float)NAN}) want(u, 0);
        for (float u : {hi + 5.0f, 2147483648.0f, 1e30f, INFINITY}) want(u, L - 2);
    }
    return bad != 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_any_coordinate_gives_a_cell_of_the_model(tmp_path):
    src, exe = tmp_path / "cells.hip", tmp_path / "cells"
    src.write_text(SRC)
    cmd = [HIPCC, "--cuda-host-only", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "emc_amd", "csrc"), str(src), "-o",
           str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[-2000:]
