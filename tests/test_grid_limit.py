"""Launches of the channel integrals on large lattices (mc_grid_limit.h), on
the host: fewer than 2^32 threads each, whatever the channels, and as many
tiles as that allows."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = r'''
#include <cstdio>
#include "mc_grid_limit.h"
int main()
{
    for (unsigned g = 1; g <= 16; ++g) std::printf("%u\n", mcb::tiles_per_launch(g));
}
'''


def test_a_launch_has_fewer_than_2_to_the_32_threads(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    (tmp_path / "limit.cpp").write_text(SRC)
    exe = str(tmp_path / "limit")
    subprocess.run([cxx, "-std=c++17", "-I", os.path.join(ROOT, "mocassin_amd", "csrc"), str(tmp_path / "limit.cpp"),
                    "-o", exe], check=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=30, check=True)
    tiles = [int(v) for v in r.stdout.split()]
    assert len(tiles) == 16                          # 64 channels, four to a wavefront
    for groups, n in enumerate(tiles, 1):
        assert n % 8 == 0 and n * groups * 64 < 2 ** 32 <= (n + 8) * groups * 64
