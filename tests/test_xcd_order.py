"""The order of workgroups over the XCDs (csrc/xcd.hpp), compiled for the host:
a bijection for every grid size, and the workgroups of one XCD (those with the
same index modulo 8) at consecutive places, also where the size is no multiple
of 8 (85 tile runs of 3 token blocks: 255)."""
import os
import subprocess

import numpy as np

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "shady_thinker_amd", "csrc")
SRC = """#include <cstdio>
#include "xcd.hpp"
int main() {
    for (int n = 1; n <= 600; ++n) {
        for (int b = 0; b < n; ++b) std::printf("%d ", st::xcd_order(b, n));
        std::printf("\\n");
    }
}
"""


def test_xcd_order(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    for n, line in enumerate(out.splitlines(), 1):
        place = np.array(line.split(), dtype=int)
        assert np.array_equal(np.sort(place), np.arange(n)), n
        for x in range(min(8, n)):
            assert np.all(np.diff(place[x::8]) == 1), (n, x)
