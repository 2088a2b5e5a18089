"""Work of more blocks than a launch holds goes out in several launches that cover it once.

The helper is plain C++ and is compiled and run here on the CPU; a launch of 2^32 threads or
more along x is refused by the runtime.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "launch_pieces.hpp"
int main(int, char** v) {
  const uint64_t units = strtoull(v[1], 0, 10), per = strtoull(v[2], 0, 10);
  brille_amd::in_pieces(units, per, [&](uint64_t first, uint64_t count, unsigned blocks) {
    printf("%llu %llu %u\n", (unsigned long long)first, (unsigned long long)count, blocks);
  });
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("pieces")
    src, exe = d / "pieces.cpp", d / "pieces"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "brille_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    return str(exe)


# a wave per vertex, 42 pairs of six modes, single pairs; up to 2^32 - 1 vertices or pairs
@pytest.mark.parametrize("per", [1, 4, 42, 256])
@pytest.mark.parametrize("units", [0, 1, 255, 256, 257, 121_200, (1 << 24) - 1, 1 << 24, 67_108_861, 67_108_864, (1 << 32) - 1])
def test_pieces_cover_the_work_once(program, units, per):
    out = subprocess.run([program, str(units), str(per)], check=True, capture_output=True, text=True).stdout
    at = 0
    for line in out.splitlines():
        first, count, blocks = map(int, line.split())
        assert first == at and count > 0 and first % per == 0
        assert blocks == -(-count // per) and blocks * 256 < 1 << 32
        at += count
    assert at == units
