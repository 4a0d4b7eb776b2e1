"""Lattices with axes so long that the walk's tables nearly fill the LDS of a
CU: packet for packet the oracle's, alone, replayed and in a batch."""
import numpy as np
import pytest

import mc_oracle as O
from test_gpu_transport import transport_from_problem

pytestmark = pytest.mark.gpu

COUNTERS = ("n_seg", "n_abs", "n_sca", "n_esc", "n_lost", "n_line", "n_trapped", "n_flights")


def _problem(nx, nb=5):
    """An octant of nx x 2 x 2 cells, thin along x, a few optical depths along y and z."""
    rng = np.random.default_rng(nx)
    w = np.float32(1e17)
    x = (np.arange(nx) * (w / 500)).astype(np.float32)
    y = np.array([0, w], np.float32)
    nc = 4 * nx
    active = np.asfortranarray(np.arange(1, nc + 1, dtype=np.int32).reshape(nx, 2, 2, order="F"))
    op = np.zeros((nc + 1, nb), np.float32, order="F")
    op[1:] = rng.uniform(0.2, 3.0, (nc, nb)).astype(np.float32) / w
    rec = np.zeros((nc + 1, nb), np.float32, order="F")
    rec[1:] = np.sort(rng.random((nc, nb)), axis=1)
    rec[1:, -1] = 1.0
    return O.Problem(xAxis=x, yAxis=y, zAxis=y, active=active, opacity=op,
                     nuArray=np.linspace(0.8, 4.0, nb).astype(np.float32),
                     specCDF=np.linspace(1.0 / nb, 1.0, nb).astype(np.float32), R_out=x[-1],
                     geoCorr=(x[1] / 2, w / 2, w / 2), ionEdge1=0.99, deltaE=1.0, starPos=(0, 0, 0), starIdx=(1, 1, 1),
                     recPDF=rec, totalLines=np.full(nc + 1, 0.2, np.float32), symmetric=True)


def _check(c, J, E, want):
    Jo, Eo, co = want
    for k in COUNTERS:
        assert c[k] == co[k], k
    assert np.allclose(J, Jo, rtol=1e-12, atol=0) and np.allclose(E, Eo, rtol=1e-12, atol=0)


# the sum of the axes up to which rings of eight fit, and beyond it the batch's thinner form
@pytest.mark.parametrize("nx", [2040, 11000, 11720])
def test_long_axes_equal_oracle(nx):
    print("axes of %d cells" % nx, flush=True)
    P = _problem(nx)
    want = P.transport(0, 500, 9, 1, O.MATH_OWN, O.J_FP64)
    rng = np.random.default_rng(1)
    d = rng.normal(size=(64, 3))
    d = (d / np.linalg.norm(d, axis=1)[:, None]).astype(np.float32)
    cell = np.stack([rng.integers(1, nx + 1, 64), np.ones(64, int), np.ones(64, int)], axis=1).astype(np.int32)
    pos = np.stack([P.xAxis[cell[:, 0] - 1], np.full(64, 1e16, np.float32), np.full(64, 2e16, np.float32)], axis=1)
    T = transport_from_problem(P, 9)
    try:
        _check(T.energy_packet_driver(1, 500, 0), *T.fetch(), want)
        seq, ds, ln, st = T.walk_replay(pos, d, cell, max_len=4096)
    finally:
        T.close()
    for i in range(64):
        oc, ods, ost = P.walk(pos[i], d[i], cell[i])
        assert ost == st[i] and np.array_equal(oc, seq[i, :ln[i]]), i
        assert np.array_equal(ods.view(np.uint32), ds[i, :ln[i]].view(np.uint32)), i


@pytest.mark.parametrize("nx", [11000, 13370])
def test_long_axes_in_a_batch_equal_oracle(nx):
    from mocassin_amd.transport import transport_batch
    print("batch with axes of %d cells" % nx, flush=True)
    probs = [_problem(nx), _problem(40)]
    models = [transport_from_problem(P, 9) for P in probs]
    try:
        cs, _ = transport_batch(models, [1, 1], [500, 700])
        for T, P, c, n in zip(models, probs, cs, (500, 700)):
            _check(c, *T.fetch(), P.transport(0, n, 9, 1, O.MATH_OWN, O.J_FP64))
    finally:
        for T in models:
            T.close()
