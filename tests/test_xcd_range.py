"""The split of a batch over workgroups: every item once, and no workgroup with
more items than the grid makes necessary (one item each when there is a
workgroup per item)."""
import os
import subprocess

from conftest import ROOT

PROGRAM = r"""
#include "xcd_range.hpp"
#include <cstdio>
#include <vector>
int main() {
    const long grids[] = {8, 9, 15, 16, 64, 1000, 2048};
    for (long n = 1; n <= 5000; n += n < 70 ? 1 : 61) {
        std::vector<long> gs(grids, grids + 7);
        gs.push_back(n);
        for (long G : gs) {
            if (G > n) continue;
            std::vector<int> seen(n, 0);
            long most = 0;
            for (long b = 0; b < G; b++) {
                const cg::XcdRange r(n, G, b);
                long count = 0;
                for (long i = r.lo; i < r.hi; i += r.step) { seen[i]++; count++; }
                if (count > most) most = count;
            }
            for (long i = 0; i < n; i++) if (seen[i] != 1) { std::printf("n %ld G %ld item %ld: %d\n", n, G, i, seen[i]); return 1; }
            const long need = (n + G - 1) / G;
            if ((G % 8 == 0 || G == n) && most > need) { std::printf("n %ld G %ld: %ld items\n", n, G, most); return 1; }
        }
    }
    return 0;
}
"""


def test_every_item_once_and_evenly(tmp_path):
    src, exe = tmp_path / "x.cpp", tmp_path / "x"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "cantera_amd", "csrc"), "-o", str(exe),
                    str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
