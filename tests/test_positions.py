"""csrc/positions.hpp, compiled for the host.

At the largest capacities (a batch's reaches 2^31 - 256) its 32-bit sums, partition
counts and ends equal 64-bit arithmetic: a position that wrapped would make a tile's
list begin before the array.  The workgroups of a raster grid name every tile once,
for chunks of any size, and XCD b % 8 gets consecutive tiles of each chunk.
"""

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


TILES = """
#include "positions.hpp"
#include <cstdio>
int main() {
    int tiles, chunk;
    while (std::scanf("%d %d", &tiles, &chunk) == 2) {
        const int grid = jsa::xcd_grid(tiles, chunk);
        std::printf("%d", grid);
        if (tiles < 100000) for (int b = 0; b < grid; ++b) std::printf(" %d", jsa::xcd_tile(b, chunk));
        else std::printf(" %d %d", jsa::xcd_tile(0, chunk), jsa::xcd_tile(grid - 1, chunk));
        std::printf("\\n");
    }
}
"""


def _build(tmp_path, source):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    (tmp_path / "main.cpp").write_text(source)
    subprocess.run([cxx, "-std=c++17", "-O2", "-fsanitize=undefined",
                    "-fno-sanitize-recover=undefined", f"-I{CSRC}", "main.cpp", "-o", "main"],
                   cwd=tmp_path, check=True)


def test_tiles_of_a_grid(tmp_path):
    _build(tmp_path, TILES)
    cases = [(n, c) for n in (1, 7, 8, 9, 63, 127, 128, 129, 1000, 8160, 10816)
             for c in sorted({1, 3, 16, 64, 100, (n + 7) // 8})]
    large = [(1 << 30, 1 << 27), (1 << 30, 64), ((1 << 30) - 5, 16)]
    out = subprocess.run([tmp_path / "main"], input="\n".join(f"{n} {c}" for n, c in cases + large),
                         text=True, capture_output=True, check=True).stdout.splitlines()
    for (n, c), line in zip(cases, out):
        grid, *tiles = map(int, line.split())
        assert grid % (8 * c) == 0 and n <= grid < n + 8 * c
        assert sorted(tiles) == list(range(grid)), (n, c)
        for x in range(8):
            own = tiles[x::8]
            assert all(b == a + 1 for i, (a, b) in enumerate(zip(own, own[1:])) if (i + 1) % c)
    for (n, c), line in zip(large, out[len(cases):]):
        grid, first, last = map(int, line.split())
        assert n <= grid < n + 8 * c and first == 0 and last == grid - 1


def test_positions_at_the_largest_capacities(tmp_path):
    _build(tmp_path, MAIN)
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
