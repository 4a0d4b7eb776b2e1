"""The hold on the deposit log (mc_hold.h): a sweep that returns on an error
waits for its stream before another sweep can take the log."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = r'''
#include <cstdio>
#include <mutex>
#include <thread>
#include "mc_hold.h"
static std::mutex m;
static int waits;
static bool held_while_waiting;
template <class F> static bool elsewhere(F f) { bool r = false; std::thread([&] { r = f(); }).join(); return r; }
static bool is_free() { return elsewhere([] { return std::unique_lock<std::mutex>(m, std::try_to_lock).owns_lock(); }); }
static int sweep(int fails_at)          // 0: never; the launches of a sweep, two rounds
{
    const auto wait = [] { ++waits; held_while_waiting = !is_free(); };
    mcl::Hold<decltype(wait)> use(wait);
    if (!use.take(m)) return 3;
    for (int round = 1, call = 0; round <= 2; ++round) {
        use.began();
        for (int k = 0; k < 4; ++k)
            if (++call == fails_at) return 1;
        use.ended();
    }
    return 0;
}
#define CHECK(x) if (!(x)) { std::printf("failed: %s\n", #x); return 1; }
int main()
{
    CHECK(sweep(0) == 0 && waits == 0 && is_free());
    for (int at = 1; at <= 8; ++at) {
        waits = 0;
        held_while_waiting = false;
        CHECK(sweep(at) == 1 && waits == 1 && held_while_waiting && is_free());
    }
    const auto never = [] { ++waits; };
    waits = 0;
    {
        mcl::Hold<decltype(never)> a(never), b(never);
        CHECK(a.take(m) && !elsewhere([&] { return b.take(m); }));
        a.drop();
        CHECK(b.take(m));
    }
    CHECK(waits == 0 && is_free());
    std::puts("ok");
}
'''


def test_a_failed_sweep_waits_before_it_lets_the_log_go(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    src = tmp_path / "hold.cpp"
    src.write_text(SRC)
    exe = str(tmp_path / "hold")
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "mocassin_amd", "csrc"), str(src),
                    "-o", exe], check=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=30)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
