"""Logged sweeps of estimators with 1.3e8 to 5.2e8 words, where all bins of
the log are in use and a bin is one, two or four ranges: against the same
sweeps with atomics.  A few of the lattice's points are cells; the packets'
segments in the others add up in row 0."""
import numpy as np
import pytest

from conftest import golden, view_from_fixture
from test_gpu_deposit import _equal, _sweep

pytestmark = pytest.mark.gpu

BINS = 7936


def _context(n, nb, nc, seed):
    """An octant of n^3 points, nc of them cells of about one optical depth."""
    from mocassin_amd import Transport
    rng = np.random.default_rng(seed)
    edge = np.float32(3e18)
    x = (np.arange(n) * (edge / (n - 1))).astype(np.float32)
    active = np.zeros(n ** 3, np.int32)
    active[rng.choice(n ** 3, nc, replace=False)] = np.arange(1, nc + 1)
    op = np.zeros((nc + 1, nb), np.float32, order="F")
    op[1:] = (10.0 ** rng.uniform(-1, 1, (nc, nb)) / (x[1] - x[0])).astype(np.float32)
    rec = np.zeros((nc + 1, nb), np.float32, order="F")
    rec[1:] = np.sort(rng.random((nc, nb)), axis=1)
    rec[1:, -1] = 1.0
    T = Transport(x, x, x, active.reshape(n, n, n, order="F"), nc, nb, np.linspace(0.8, 4.0, nb).astype(np.float32),
                  edge, (x[1] / 2,) * 3, 0.5, [(0.0, 0.0, 0.0)], [(1, 1, 1)], [1.0], symmetric=True, seed=seed)
    T.upload_tables(op, np.linspace(1.0 / nb, 1.0, nb).astype(np.float32).reshape(-1, 1), rec,
                    np.full(nc + 1, 0.3, np.float32))
    return T


# nearly all bins of one range; just beyond, two ranges a bin (and three escape
# planes); just beyond that, four; nearly all bins of four, the most words
@pytest.mark.parametrize("n,nb,nc,views,shift", [(120, 75, 1000, False, 14), (120, 75, 20000, False, 15),
                                                 (116, 80, 23000, True, 15), (120, 150, 20000, False, 16),
                                                 (120, 300, 4000, False, 16)])
def test_logged_sweep_of_many_words_equals_atomics(n, nb, nc, views, shift):
    view = view_from_fixture(golden("transport_c1mini_view")) if views else None
    words = n ** 3 * nb + (nc + 1) * (nb + 1) * (3 if views else 1)
    assert BINS << (shift - 1) < words <= BINS << shift or shift == 14
    T = _context(n, nb, nc, 77 + nb)
    try:
        if views:
            T.set_view_angles(view)
        per = T.energy_packet_driver(1, 20000, 0)["n_seg"] / 20000.0
        packets = int(1.2 * (3e6 + 0.2 * words) / per) + 1
        print("log of %.3g words, %d packets of %.1f segments" % (words, packets, per), flush=True)
        _equal(_sweep(T, "auto", packets), _sweep(T, "one", packets), packets)
    finally:
        T.close()
