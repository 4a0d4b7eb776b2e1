"""A state on its way to the device: laid out there, in one pinned piece or
several, from two threads at once, against the same cells a few hundred at a
time, which are laid out on the host."""
import threading

import numpy as np
import pytest

from conftest import balance_fixture
from test_gpu_opacity_bins import _lattice

pytestmark = pytest.mark.gpu


def _setup(n, b):
    T = _lattice(n, b)
    T.balance_setup(b)
    rng = np.random.default_rng(3)
    segs = [[z, ion, 2 + z, b.nbins - ion] for z in range(1, 31) if b.elem_on[z - 1]
            for ion in range(1, min(z, b.nstages) + 1)]
    T.opacity_setup(segs, 10.0 ** rng.uniform(-3, 0, sum(s[3] - s[2] + 1 for s in segs)).astype(np.float32), 1e-3)
    return T


def _state(rows, b, seed):
    rng = np.random.default_rng(seed)
    return (rng.uniform(10, 1000, rows).astype(np.float32), rng.uniform(5e3, 2e4, rows).astype(np.float32),
            rng.uniform(10, 1000, rows).astype(np.float32),
            (10.0 ** rng.uniform(-6, 0, (rows, b.nElemUsed, b.nstages))).astype(np.float32))


# 38 words a cell: one piece of 4 MiB, two and four
@pytest.mark.parametrize("n", [29, 50, 68])
def test_large_states_arrive_whole(n):
    b = balance_fixture("c2mini")[0]
    T = [_setup(n, b) for _ in range(2)]
    rows = T[0].nCells + 1
    print("state of %d cells" % (rows - 1), flush=True)
    states = [_state(rows, b, seed) for seed in (1, 2)]
    got = [[], []]

    def build(k):
        for _ in range(3):
            got[k].append(T[k].opacity_build(*states[k])[0])
    try:
        th = [threading.Thread(target=build, args=(k,)) for k in range(2)]
        for t in th:
            t.start()
        for t in th:
            t.join()
    finally:
        for t in T:
            t.close()
    small = _setup(12, b)                  # 576 cells
    few = small.nCells + 1
    assert few * 45 * 8 <= 256 << 10
    try:
        for k in range(2):
            assert len(got[k]) == 3 and all(np.array_equal(g, got[k][0]) for g in got[k])
            for first in (1, rows // 2, rows - few + 1):
                cells = np.r_[0, first:first + few - 1]
                want = small.opacity_build(*(v[cells] for v in states[k]))[0]
                assert np.array_equal(got[k][0][cells][1:].view(np.uint32), want[1:].view(np.uint32))
    finally:
        small.close()


# either side of the rows that are laid out on the host (256 KB: 728 cells)
def test_rows_of_host_and_device_are_the_same():
    b = balance_fixture("c2mini")[0]
    got = []
    for n in (12, 13):                     # 576 and 732 cells
        print("state of a %d^3 lattice" % n, flush=True)
        T = _setup(n, b)
        try:
            assert (T.nCells + 1) * 45 * 8 <= 256 << 10 if n == 12 else (T.nCells + 1) * 45 * 8 > 256 << 10
            state = [v[:T.nCells + 1] for v in _state(2000, b, 5)]
            got.append((T.opacity_build(*state)[0], T.line_luminosities(*state)[0]))
        finally:
            T.close()
    few = len(got[0][0])
    assert np.array_equal(got[0][0].view(np.uint32), got[1][0][:few].view(np.uint32))
    assert all(np.isfinite(f).all() and (f > 0).any() for _, f in got)
