"""The grain terms of the balance over the row counts where their layout
changes (one row on all 64 lanes to 32 rows on two lanes each) and over
thresholds at its edges: below the first frequency bin, on a bin, above the
last.  Against the FP64 restatement, with the bound of the deck's own rows
(sums in another order: 1e-9)."""
import numpy as np
import pytest

import mc_oracle as O
from test_gpu_dust import _context, _fixture, _oracle_dict, _pe_tables

pytestmark = pytest.mark.gpu


# the photoelectric threshold of each species (Ryd); "bin" is a mesh frequency
@pytest.mark.parametrize("nSz,vn", [
    (1, [0.588]), (2, [0.588]), (1, [0.588, 0.4, 0.9]), (5, [0.45]), (3, ["bin", 30.0, 1e-7]),
    (17, [0.588]), (8, [0.588, "bin", 0.35, 2.0]),
])
def test_grain_rows_match_oracle(nSz, vn):
    print("grain rows", nSz, vn, flush=True)
    f, b, J, Hden, Te0, Ne0, ion0, _, _, _ = _fixture("dust_pe")
    nS, nT, nc1, nb = len(vn), 1500, J.shape[0], b.nbins
    rng = np.random.default_rng(nS * 100 + nSz)
    rows = f["dust_abs"].reshape(-1, nb)
    absx = np.array([[rows[(3 * s + a) % len(rows)] * rng.uniform(0.5, 2.0) for a in range(nSz)] for s in range(nS)],
                    np.float32)
    t = np.arange(1, nT + 1, dtype=np.float64)
    em = (rng.uniform(0.5, 2.0, (nS, nSz, 1)) * 1e-9 * t ** 5).astype(np.float32)
    g = _oracle_dict(absx, rng.dirichlet(np.ones(nSz)).astype(np.float32), rng.dirichlet(np.ones(nS)).astype(np.float32),
                     em, nS)
    g.update(dust_vn=np.array([b.nuArray[127] if v == "bin" else v for v in vn], np.float32),
             dust_msurf=rng.uniform(12.0, 30.0, nS).astype(np.float32),
             dust_radius=np.geomspace(0.005, 0.25, nSz).astype(np.float32),
             dust_aweight=f["dust_aweight"], dust_ndust=f["dust_ndust"])
    T0 = rng.uniform(10.0, 100.0, (nc1, nSz + 1, nS + 1))
    cells = np.arange(1, nc1)[::4]
    T = _context(nc1 - 1, nb, b.nuArray)
    try:
        T.set_estimators(J.astype(np.float64))
        T.balance_setup(b)
        T.dust_setup(**_pe_tables(g))
        Tg, fl, nI, _, Te, Ne, ion = T.update_grains(T0, Hden=Hden, Te=Te0, Ne=Ne0, ionDen=ion0)
    finally:
        T.close()
    Teo, Neo, iono, flo, nIo, gdc, peh, _ = O.Balance(b).run_grains(J.astype(np.float64), Hden, Te0, Ne0, ion0, g, T0,
                                                                    "f64", cells=cells)
    To = O.dust_temps(J.astype(np.float64), T0, g, "f64", gdc=gdc, peh=peh)
    c = cells
    assert np.array_equal(fl[c], flo[c]) and np.array_equal(nI[c], nIo[c])
    assert np.max(np.abs(Te[c] - Teo[c]) / Teo[c]) < 1e-9
    assert np.max(np.abs(Ne[c] - Neo[c]) / Neo[c]) < 1e-9
    on = iono[c] > 0
    assert np.max(np.abs(ion[c][on] - iono[c][on]) / iono[c][on]) < 1e-8
    assert np.max(np.abs(Tg[c] - To[c]) / To[c].clip(1)) < 1e-9
