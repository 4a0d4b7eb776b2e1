"""Which sweeps the deposit log is for and how it divides their words
(mc_log_shape.h), on the host: the sizes where the division changes, and the
side of the line on which sweeps lie whose two forms were timed more than a
tenth apart."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = r'''
#include <cstdio>
#include <cstdlib>
#include "mc_log_shape.h"
int main(int argc, char **argv)
{
    for (int i = 1; i < argc; ++i) {
        const mcl::Shape s = mcl::shape(std::strtoull(argv[i], nullptr, 10));
        std::printf("%u %d %d %.17g\n", s.words, s.shift, s.bins, mcl::least_deposits(s));
    }
}
'''


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("shape")
    (d / "shape.cpp").write_text(SRC)
    exe = str(d / "shape")
    subprocess.run([cxx, "-std=c++17", "-I", os.path.join(ROOT, "mocassin_amd", "csrc"), str(d / "shape.cpp"), "-o", exe],
                   check=True, timeout=120)

    def run(words):
        r = subprocess.run([exe] + [str(int(w)) for w in words], capture_output=True, text=True, timeout=30, check=True)
        return [[float(v) for v in line.split()] for line in r.stdout.splitlines()]
    return run


def test_words_of_a_bin_double_where_the_bins_run_out(shapes):
    B = 7936
    words = [0, 1, 16384, 16385, B << 14, (B << 14) + 1, B << 15, (B << 15) + 1, B << 16, (B << 16) + 1]
    want = [(0, 14, 0), (1, 14, 1), (16384, 14, 1), (16385, 14, 2), (B << 14, 14, B), ((B << 14) + 1, 15, B // 2 + 1),
            (B << 15, 15, B), ((B << 15) + 1, 16, B // 2 + 1), (B << 16, 16, B), (0, 14, 0)]
    assert [tuple(s[:3]) for s in shapes(words)] == want


def test_sweeps_take_the_faster_side(shapes):
    logged = [(9.5e5, 8e6), (3.2e5, 4e6), (4.8e6, 1.6e7), (1.9e7, 3.2e7), (6.3e7, 3.2e7), (2.3e8, 1e8), (8.7e7, 1e8)]
    atomics = [(4.1e8, 4e6), (4.1e8, 3.2e7), (3.1e8, 3.2e7), (2.3e8, 8e6), (1.8e8, 8e6), (6.3e7, 4e6), (1.3e8, 1.6e7)]
    for on, sweeps in ((True, logged), (False, atomics)):
        for (words, deposits), s in zip(sweeps, shapes([w for w, _ in sweeps])):
            assert (deposits >= s[3]) == on, (words, deposits, s)
