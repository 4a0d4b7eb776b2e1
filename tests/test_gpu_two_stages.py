"""The balance with two ionisation stages, the least: there is no He++, whose
cooling terms are zero.  Against the FP64 restatement."""
import numpy as np
import pytest

import mc_oracle as O
from conftest import balance_fixture
from test_gpu_balance import _context
from test_gpu_balance_lanes import _subset

pytestmark = pytest.mark.gpu


# H and He (4 lanes a cell), and with the metals of the deck (16)
@pytest.mark.parametrize("z_on", [[1, 2], [1, 2, 6, 7, 8, 10, 16]])
def test_two_stages_equal_oracle(z_on):
    print("two stages, elements", z_on, flush=True)
    b, J, Hden, Te0, Ne0, ion0, _ = balance_fixture("c2mini")
    b, ion0 = _subset(b, ion0, z_on)
    b.nstages, ion0 = 2, np.ascontiguousarray(ion0[:, :, :2])
    J = J.astype(np.float64)
    T = _context(J.shape[0] - 1, b.nbins, b.nuArray)
    try:
        T.balance_setup(b)
        T.set_estimators(J)
        Te, Ne, ion, fl, nT, _ = T.update_cells(Hden, Te0, Ne0, ion0)
    finally:
        T.close()
    Te_o, Ne_o, ion_o, fl_o, nT_o = O.Balance(b).run(J, Hden, Te0, Ne0, ion0, "f64")
    c = slice(1, None)
    assert ((fl[c] & 16) == 0).sum() > 50
    assert np.array_equal(fl[c], fl_o[c]) and np.array_equal(nT[c], nT_o[c])
    assert np.max(np.abs(Te[c] - Te_o[c]) / Te_o[c]) < 1e-9
    assert np.max(np.abs(Ne[c] - Ne_o[c]) / Ne_o[c]) < 1e-9
    assert np.max(np.abs(ion[c] - ion_o[c]) / ion_o[c].clip(1e-15)) < 1e-8
