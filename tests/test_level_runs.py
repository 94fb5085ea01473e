"""The split of an element's levels into runs (nekcem_amd/csrc/level_runs.hpp),
compiled for the host: at every order and slab count the runs cover the levels
once, and every slot of every run, the dropped last one of a short run among
them, stands for a level of the element, so that its row of the derivative
matrix lies in the kernels' table."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "nekcem_amd", "csrc")

SRC = r"""
#include <cstdio>
#include "level_runs.hpp"
using namespace nkc;
int main() {
    int seen = 0, shorts = 0;
    for (int n1 = 4; n1 <= 10; ++n1)
        for (int sl = 1; sl <= 5; ++sl) {
            if (sl > 1 && !slabs_built(n1, sl)) continue;
            const int runs = level_runs(n1) * sl, KL = run_length(n1, sl);
            ++seen;
            for (int run = 0, next = 0; run < runs; ++run) {
                const int k0 = next, kn = n1 / runs + (run < n1 % runs);
                next += kn;
                if ( kn < 1 || kn > KL || kn < KL - 1 || (run == runs - 1 && k0 + kn != n1))
                    return printf("run %d of %d at n1 = %d: %d + %d\n", run, runs, n1, k0, kn), 1;
                shorts += kn < KL;
                for (int kk = 0; kk < KL; ++kk) {
                    const int k = slot_level(n1, runs, k0, kn, kk);
                    if (k < 0 || k >= n1 || (kk < kn && k != k0 + kk))
                        return printf("slot %d of run %d of %d at n1 = %d: level %d\n", kk, run, runs, n1, k), 1;
                }
            }
        }
    printf("%d %d\n", seen, shorts);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_slot_is_a_level(tmp_path):
    (tmp_path / "runs.cpp").write_text(SRC)
    exe = str(tmp_path / "runs")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-o", exe, str(tmp_path / "runs.cpp")],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    seen, shorts = map(int, r.stdout.split())
    assert seen >= 7 and shorts > 0      # whole elements of every order, and runs of unequal length
