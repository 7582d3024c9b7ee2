"""The split of launches that a HIP grid (fewer than 2^32 work-items) cannot hold: host arithmetic of csrc/grid.hpp,
compiled by the host compiler, at the sizes where it starts and far beyond any that the tests could run."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "octrees-benchmark_amd", "csrc")
PROGRAM = r"""
#include "grid.hpp"
#include <cstdio>
#include <cstdlib>
int main(int argc, char **argv) {
    const size_t blocks = strtoull(argv[1], 0, 10), threads = strtoull(argv[2], 0, 10);
    oct::for_grids(blocks, threads, [](uint32_t first, unsigned n) { printf("%u %u\n", first, n); });
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("grid")
    (d / "grid.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(d / "grid.cpp"), "-o", str(d / "grid")], check=True)
    return str(d / "grid")


@pytest.mark.parametrize("threads", [64, 256])
@pytest.mark.parametrize("items", [0, 1, 2**32 - 257, 2**32 - 256, 2**32 - 1, 2**32, 2**33 + 5, 3 * (2**32 - 256), 2**36])
def test_ranges_cover_the_launch(program, items, threads):
    blocks = -(-items // threads)
    out = subprocess.run([program, str(blocks), str(threads)], check=True, capture_output=True, text=True).stdout
    at = 0
    for line in out.splitlines():
        first, n = map(int, line.split())
        assert first == at and 0 < n and n * threads < 2**32
        at += n
    assert at == blocks
    assert len(out.splitlines()) == -(-blocks // ((2**32 - 1) // threads))
