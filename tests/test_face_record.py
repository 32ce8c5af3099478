"""The word that links the two records of a face (csrc/face_record.hpp) keeps
every index it can be given, also above 2^29: a mesh has up to four records
per cell, so their numbers go past those of its cells.  Compiled for the host."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "netflux_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "face_record.hpp"
int main(int argc, char **argv) {
    for (int q = 1; q < argc; ++q)
        for (int f = 0; f < 4; ++f) {
            const uint32_t w = nf::rec_word(f & 1, f & 2, (uint32_t)std::strtoul(argv[q], nullptr, 10));
            std::printf("%u %d %d\n", nf::rec_index(w), (w & nf::REC_BOUNDARY) != 0, (w & nf::REC_OWNER) != 0);
        }
    std::printf("%llu\n", (unsigned long long)nf::REC_MAX);
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("face_record")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", d / "main", d / "main.cpp"], check=True)
    return d / "main"


def test_every_index_comes_back(program):
    idx = [0, 1, 2**28, 2**29 - 1, 2**29, 2**29 + 1, 3 * 2**28 + 5, 2**30 - 1]
    out = subprocess.run([program] + [str(i) for i in idx], check=True, capture_output=True, text=True).stdout.split("\n")
    got = [tuple(map(int, line.split())) for line in out[:4 * len(idx)]]
    assert got == [(i, f & 1, f >> 1) for i in idx for f in range(4)]
    assert int(out[4 * len(idx)]) == 2**30  # records beyond it keep the sweeps that gather per lane
