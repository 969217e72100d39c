"""csrc/positions.hpp at the largest capacities (a batch's reaches 2^31 - 256): its
32-bit sums, partition counts and ends against 64-bit arithmetic, compiled for the
host.  A position that wrapped would make a tile's list begin before the array."""

import itertools
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "jaxsplat_amd" / "csrc"
MAIN = """
#include "positions.hpp"
#include <cstdio>
int main() {
    int a, cap, size;
    unsigned b;
    while (std::scanf("%d %u %d %d", &a, &b, &cap, &size) == 4)
        std::printf("%d %d %d\\n", jsa::clamped_sum(a, b, cap),
                    jsa::part_count(a < (int)b ? a : (int)b, cap, size),
                    jsa::part_end(a, cap, size));
}
"""


def test_positions_at_the_largest_capacities(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    (tmp_path / "main.cpp").write_text(MAIN)
    subprocess.run([cxx, "-std=c++17", "-O2", "-fsanitize=undefined",
                    "-fno-sanitize-recover=undefined", f"-I{CSRC}", "main.cpp", "-o", "main"],
                   cwd=tmp_path, check=True)
    cases = []
    for cap in (1, 1023, 1024, 1025, (1 << 30) - 1, (1 << 30) + 7, 0x7FFFFF00 - 1, 0x7FFFFF00):
        at = sorted({min(v, cap) for v in (0, 1, 1023, 1024, 1 << 29, 1 << 30, cap - 1024,
                                           cap - 1023, cap - 1, cap) if v >= 0})
        cases += [(a, b, cap, 1024) for a, b in itertools.product(at, at) if a < cap]
    out = subprocess.run([tmp_path / "main"], input="\n".join(" ".join(map(str, c)) for c in cases),
                         text=True, capture_output=True, check=True).stdout.split()
    got = [tuple(map(int, out[i:i + 3])) for i in range(0, len(out), 3)]
    want = [(min(a + b, cap), -(-(cap - min(a, b)) // size), min(cap, a + size))
            for a, b, cap, size in cases]
    assert got == want
