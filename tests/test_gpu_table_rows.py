"""Table rows of a lattice that lacks a cell: its row is zero, whatever the
device's memory held before."""
import numpy as np
import pytest

from mocassin_amd import _capi

pytestmark = pytest.mark.gpu


def _context(active, nc, nb):
    from mocassin_amd import Transport
    n = active.shape[0]
    x = (np.arange(n) * 1e17).astype(np.float32)
    T = Transport(x, x, x, np.asfortranarray(active), nc, nb, np.linspace(0.8, 4.0, nb).astype(np.float32), x[-1],
                  (5e16,) * 3, 0.5, [(0.0, 0.0, 0.0)], [(1, 1, 1)], [1.0], symmetric=True, seed=1)
    op = np.zeros((nc + 1, nb), np.float32, order="F")
    op[1:] = np.random.default_rng(nc).uniform(1e-18, 2e-18, (nc, nb))
    rec = np.zeros((nc + 1, nb), np.float32, order="F")
    rec[1:] = np.linspace(1.0 / nb, 1.0, nb)
    T.upload_tables(op, np.linspace(1.0 / nb, 1.0, nb).astype(np.float32).reshape(-1, 1), rec,
                    np.zeros(nc + 1, np.float32))
    return T, op


@pytest.mark.parametrize("n,nb", [(5, 65), (6, 400)])
def test_rows_without_a_lattice_point_are_zero(n, nb):
    print("table rows", n, nb, flush=True)
    nc = n ** 3
    whole = np.arange(1, nc + 1, dtype=np.int32).reshape((n, n, n), order="F")
    gone = [2, nc // 2, nc]
    cut = np.where(np.isin(whole, gone), 0, whole).astype(np.int32)
    for active in (whole, cut):                  # the first leaves its rows in the memory that the second gets
        T, op = _context(active, nc, nb)
        try:
            rows = T._rows(_capi.MC_TABLE_OPACITY)
        finally:
            T.close()
        want = op.copy()
        if active is cut:
            want[gone] = 0.0
        assert np.array_equal(rows, want)
