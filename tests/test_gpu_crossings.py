"""Crossing counts cell by cell: packets in a lattice without opacity cross a
cell at most once, so the oracle's J of each packet alone says which."""
import numpy as np
import pytest

import mc_oracle as O
from test_gpu_transport import transport_from_problem

pytestmark = pytest.mark.gpu

SIZE, BINS, PACKETS = (9, 10, 13), 5, 300


def _problem(src):
    rng = np.random.default_rng(4)
    axes = [np.cumsum(rng.uniform(0.5, 1.5, n)).astype(np.float32) * np.float32(1e17) for n in SIZE]
    nc = int(np.prod(SIZE))
    rec = np.zeros((nc + 1, BINS), np.float32, order="F")
    rec[1:] = np.linspace(1.0 / BINS, 1.0, BINS)
    # inside its cell, off the axis values
    pos = [0.5 * a[i - 1] + 0.25 * (a[max(i - 2, 0)] + a[min(i, n - 1)]) for a, i, n in zip(axes, src, SIZE)]
    return O.Problem(xAxis=axes[0], yAxis=axes[1], zAxis=axes[2],
                     active=np.asfortranarray(np.arange(1, nc + 1, dtype=np.int32).reshape(SIZE, order="F")),
                     opacity=np.zeros((nc + 1, BINS), np.float32, order="F"),
                     nuArray=np.linspace(1.1, 4.0, BINS).astype(np.float32),
                     specCDF=np.linspace(1.0 / BINS, 1.0, BINS).astype(np.float32), R_out=0.0,
                     geoCorr=(1e16, 1e16, 1e16), ionEdge1=0.99, deltaE=1.0, starPos=pos, starIdx=src, recPDF=rec,
                     totalLines=np.full(nc + 1, 0.2, np.float32), symmetric=False)


# the source in the first tile, in a middle one and in the last, which the lattice's end cuts
@pytest.mark.parametrize("src", [(1, 2, 1), (5, 6, 8), (9, 10, 13)])
@pytest.mark.parametrize("kernel", ["auto", "one", "batch"])
def test_crossings_of_every_cell_equal_oracle(src, kernel):
    print("crossings from", src, kernel, flush=True)
    P = _problem(src)
    want = np.zeros(P.nCells + 1, np.int64)
    segments = 0
    for i in range(2 * PACKETS):
        J, _, c = P.transport(i, 1, 21, 1, O.MATH_OWN, O.J_FP64)
        want += (J > 0).any(axis=1)
        segments += c["n_seg"]
    assert want.sum() == segments
    T = transport_from_problem(P, 21)
    try:
        T.count_crossings(True)
        for first in (0, PACKETS):
            if kernel == "batch":
                from mocassin_amd.transport import transport_batch
                transport_batch([T], [1], [PACKETS], [first])
            else:
                T.set_tuning(kernel=kernel)
                T.energy_packet_driver(1, PACKETS, first)
        assert np.array_equal(T.crossings(), want)
    finally:
        T.close()
