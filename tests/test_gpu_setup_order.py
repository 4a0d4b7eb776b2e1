"""Opacity and re-emission tables of one set of elements after a set-up of the
balance with another: refused where the new rows do not hold their ions, the
same tables where they do."""
import numpy as np
import pytest

from conftest import balance_fixture, golden, grid_from_fixture
from mocassin_amd import _capi
from mocassin_amd.atomic import emission_tables
from test_gpu_balance_lanes import _subset
from test_gpu_opacity import _segments

pytestmark = pytest.mark.gpu


def test_tables_of_other_elements_are_refused():
    from mocassin_amd.transport import Transport
    print("set-up order", flush=True)
    g = golden("opacity_c2mini")
    b, _, _, _, _, ion0, _ = balance_fixture("c2mini")
    two = _subset(b, ion0, [1, 2])[0]
    axes, active, nc, nb, fl, star_idx = grid_from_fixture(g)
    ion = g["ionDen"].reshape(b.nstages, b.nElemUsed, nc + 1).transpose(2, 1, 0)
    state = (g["Hden"], g["Te"], g["Ne"])
    T = Transport(*axes, active, nc, nb, b.nuArray, R_out=float(axes[0][-1]), geoCorr=(0, 0, 0), ionEdge1=1.0,
                  starPos=(0, 0, 0), starIdx=star_idx, deltaE=1.0, symmetric=fl["symmetric"], gas=True)
    try:
        T.balance_setup(b)
        T.opacity_setup(*_segments(g))
        T.emission_setup(**emission_tables(g))
        op, rec = T.opacity_build(*state, ion)[0], T.emission_build(*state, ion)[0]
        T.balance_setup(b)                               # the same elements again
        assert np.array_equal(T.opacity_build(*state, ion)[0], op)
        assert np.array_equal(T.emission_build(*state, ion)[0], rec)
        T.balance_setup(two)
        ion2 = np.ascontiguousarray(ion[:, :2, :])
        with pytest.raises(_capi.McError, match="mc_opacity_setup"):
            T.opacity_build(*state, ion2)
        with pytest.raises(_capi.McError, match="mc_emission_setup"):
            T.emission_build(*state, ion2)
    finally:
        T.close()
