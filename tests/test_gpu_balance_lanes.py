"""The balance without model ions, where a cell has 4 or 16 lanes of a
wavefront or all 64: element sets on either side of each line, cell counts
that leave the last wavefront part empty, and cells that no packet reached
beside others.  Against the FP64 restatement."""
import copy

import numpy as np
import pytest

import mc_oracle as O
from conftest import balance_fixture
from test_gpu_balance import _context

pytestmark = pytest.mark.gpu


def _subset(b, ion0, z_on):
    """The bundle with the elements z_on alone and no model ions."""
    b = copy.copy(b)
    cols = [int(b.xref[z - 1]) - 1 for z in z_on]
    b.elem_on = np.array([1 if z in z_on else 0 for z in range(1, 31)], b.elem_on.dtype)
    b.xref = np.array([z_on.index(z) + 1 if z in z_on else 0 for z in range(1, 31)], b.xref.dtype)
    b.nElemUsed = len(z_on)
    keep = np.isin(b.ch_meta[:, 0], z_on)
    b.ch_meta, b.ch_sigma = b.ch_meta[keep], np.ascontiguousarray(b.ch_sigma[keep])
    b.nch = int(keep.sum())
    b.ncel = 0
    b.cel_meta, b.cel_dbl, b.cel_flt = np.zeros((0, 6), np.int32), np.zeros(0), np.zeros(0, np.float32)
    return b, np.ascontiguousarray(ion0[:, cols, :])


# 3 channels (4 lanes), 7 to 15 (16 lanes), 19 (64 lanes)
@pytest.mark.parametrize("z_on,cells", [([1, 2], 16), ([1, 2], 33), ([1, 2, 6], 5), ([1, 2, 6, 7], 30),
                                        ([1, 2, 6, 7, 8], 7), ([1, 2, 6, 7, 8, 10], 9)])
def test_cells_side_by_side_equal_oracle(z_on, cells):
    b, J, Hden, Te0, Ne0, ion0, _ = balance_fixture("c2mini")
    b, ion0 = _subset(b, ion0, z_on)
    # the first cells of the deck, and some no packet reached among them
    pick = np.concatenate([[0], 1 + np.arange(cells) * ((J.shape[0] - 1) // cells)])
    J, Hden, Te0, Ne0, ion0 = J[pick].astype(np.float64), Hden[pick], Te0[pick], Ne0[pick], ion0[pick]
    J[2::7] = 0.0
    print("balance of %d channels, %d cells" % (b.nch, cells), flush=True)
    T = _context(cells, b.nbins, b.nuArray)
    try:
        T.balance_setup(b)
        T.set_estimators(J)
        Te, Ne, ion, fl, nT, _ = T.update_cells(Hden, Te0, Ne0, ion0)
        # a second call takes the cells in another order
        again = T.update_cells(Hden, Te0, Ne0, ion0)
    finally:
        T.close()
    for x, y in zip((Te, Ne, ion, fl, nT), again):
        assert np.array_equal(x, y)
    Te_o, Ne_o, ion_o, fl_o, nT_o = O.Balance(b).run(J, Hden, Te0, Ne0, ion0, "f64")
    c = slice(1, None)
    assert np.array_equal(fl[c], fl_o[c]) and np.array_equal(nT[c], nT_o[c])
    assert ((fl[c] & 16) == 0).sum() > cells // 2
    assert np.max(np.abs(Te[c] - Te_o[c]) / Te_o[c]) < 1e-9
    assert np.max(np.abs(Ne[c] - Ne_o[c]) / Ne_o[c]) < 1e-9
    big = ion_o[c] > 1e-15
    assert np.max(np.abs(ion[c][big] - ion_o[c][big]) / ion_o[c][big]) < 1e-8
