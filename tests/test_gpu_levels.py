"""The n-level solves (four model ions to a wavefront) at the sizes where
their layout changes, through the line luminosities: 2 to 17 levels, one,
two and more temperatures, inside and outside the tables, full and partly
filled batches, with and without level recombination, against the oracle's
FP64 restatement."""
import copy

import numpy as np
import pytest

import mc_oracle as O
from conftest import balance_fixture, golden, grid_from_fixture

pytestmark = pytest.mark.gpu


def _ions(rng, levels, temps):
    """cel_meta, cel_dbl and cel_flt of made-up ions of the fixture's elements."""
    where = [(6, 1), (6, 2), (6, 3), (7, 1), (7, 2), (8, 1), (8, 2), (8, 3), (16, 2)]
    meta, dbl, flt = [], [], []
    for k, (nl, nt) in enumerate(zip(levels, temps)):
        z, ion = where[k]
        e = np.concatenate([[0.0], np.cumsum(rng.uniform(20.0, 9000.0, nl - 1))])
        a = np.zeros((nl, nl))
        q = np.zeros((nt, nl, nl))
        for lo in range(nl):
            for up in range(lo + 1, nl):
                if (lo, up) == (0, 1) or rng.random() < 0.6:
                    a[up, lo] = 10.0 ** rng.uniform(-6, 1)
                q[:, lo, up] = rng.uniform(0.1, 4.0) * rng.uniform(0.8, 1.2, nt)
        meta.append([z, ion, 1, 2, nl, nt])
        dbl += [e, a.ravel(order="F"), q.ravel(order="F")]
        logt = np.linspace(3.5, 4.2, nt) if nt > 1 else np.array([4.0])
        br = 1.0 if k % 3 == 0 else 0.0
        flt += [logt, 2.0 * rng.integers(0, 4, nl) + 1.0, [br, float(ion)], [5.0, -0.6, 0.2, 0.7],
                [0.1, 0.3, -0.05, 0.01, 0.4]]
    return (np.array(meta, np.int32).reshape(-1, 6), np.concatenate(dbl), np.concatenate(flt).astype(np.float32))


# one small batch of one; the 8-row form's edge; both forms with a batch left
# part empty; the largest ions; one to three temperatures and a long table
@pytest.mark.parametrize("levels,temps", [
    ((2,), (3,)),
    ((9, 8, 3, 2), (5, 1, 2, 3)),
    ((10, 9, 2, 2, 9), (4, 4, 1, 2, 23)),
    ((17, 17, 16, 15, 17, 5), (23, 3, 2, 1, 4, 7)),
    ((13, 2, 17, 4, 10, 6, 9, 12, 3), (3, 1, 2, 64, 4, 5, 23, 2, 3)),
])
def test_level_solves_equal_oracle(levels, temps):
    from mocassin_amd.transport import Transport
    print("levels", levels, temps, flush=True)
    g = golden("opacity_c2mini")
    b = copy.copy(balance_fixture("c2mini")[0])
    b.cel_meta, b.cel_dbl, b.cel_flt = _ions(np.random.default_rng(len(levels)), levels, temps)
    b.ncel = len(levels)
    axes, active, nc, nb, fl, star_idx = grid_from_fixture(g)
    ion = g["ionDen"].reshape(b.nstages, b.nElemUsed, nc + 1).transpose(2, 1, 0).copy()
    ion[3] = 0.0                                      # up = 0/0: no emission from this cell
    Te = g["Te"].copy()
    Te[1], Te[2] = 2500.0, 25000.0                    # below and above the tables
    T = Transport(*axes, active, nc, nb, b.nuArray, R_out=float(axes[0][-1]), geoCorr=(0, 0, 0),
                  ionEdge1=1.0, starPos=(0, 0, 0), starIdx=star_idx, deltaE=1.0,
                  symmetric=fl["symmetric"], gas=True)
    try:
        T.balance_setup(b)
        forb, hb, _ = T.line_luminosities(g["Hden"], Te, g["Ne"], ion)
    finally:
        T.close()
    dV, cells = O.cell_volumes(*axes, active, fl["symmetric"])
    ex, _ = O.Balance(b).line_lum(g["Hden"], Te, g["Ne"], ion, dV, cells, "f64")
    assert forb.shape == ex.shape and np.all(np.isfinite(ex)) and np.any(ex > 0)
    assert np.array_equal(forb == 0, ex == 0)
    # the bound of the line luminosities on the reference's ions
    big = ex != 0
    assert np.max(np.abs(forb[big] / ex[big] - 1)) < 1e-7
