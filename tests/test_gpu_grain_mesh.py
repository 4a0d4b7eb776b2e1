"""The balance with grains on meshes of up to the 4096 bins that the grains
take, where the LDS of four cells side by side would not fit a CU: against
the FP64 restatement, with the bound of the deck's own mesh (sums in another
order: 1e-9)."""
import copy

import numpy as np
import pytest

import mc_oracle as O
from test_gpu_dust import _context, _fixture, _oracle_dict, _pe_tables

pytestmark = pytest.mark.gpu


def _on_mesh(nb, nSz, seed=0):
    """The dust deck on nb bins with nSz grain sizes of one species: tables
    and J between the deck's bins, its edges at the bin they fall in."""
    f, b, J, Hden, Te0, Ne0, ion0, _, _, _ = _fixture("dust_pe")
    rng = np.random.default_rng(seed)
    x = b.nuArray.astype(np.float64)
    nu = np.interp(np.linspace(0, x.size - 1, nb), np.arange(x.size), x).astype(np.float32)
    on = lambda a: np.array([np.interp(nu, x, r) for r in np.reshape(a, (-1, x.size))])
    rows = on(f["dust_abs"])
    b = copy.copy(b)
    b.ch_sigma = on(b.ch_sigma).astype(np.float32)
    b.ch_meta = b.ch_meta.copy()
    b.ch_meta[:, 4:7] = np.minimum(np.searchsorted(nu, x[b.ch_meta[:, 4:7] - 1] * (1 - 1e-6)) + 1, nb)
    b.nuArray, b.nbins = nu, nb
    absx = np.array([[rows[a % len(rows)] * rng.uniform(0.5, 2.0) for a in range(nSz)]], np.float32)
    em = (rng.uniform(0.5, 2.0, (1, nSz, 1)) * 1e-9 * np.arange(1, 1501, dtype=np.float64) ** 5).astype(np.float32)
    g = _oracle_dict(absx, rng.dirichlet(np.ones(nSz)).astype(np.float32), np.ones(1, np.float32), em, 1)
    g.update(dust_vn=np.array([0.588], np.float32), dust_msurf=np.array([20.0], np.float32),
             dust_radius=np.geomspace(0.005, 0.25, nSz).astype(np.float32), dust_aweight=f["dust_aweight"],
             dust_ndust=f["dust_ndust"])
    J = on(J) * (x.size / nb)
    T0 = rng.uniform(10.0, 100.0, (J.shape[0], nSz + 1, 2))
    return b, J, (Hden, Te0, Ne0, ion0), g, T0


def _with_elements(b, ion0, z_on, ns):
    """The bundle with elements z_on (H and He first) and ns stages; those the
    deck lacks are neutral, without photoionisation."""
    b = copy.copy(b)
    b.elem_on = np.array([1 if z in z_on else 0 for z in range(1, 31)], b.elem_on.dtype)
    b.xref = np.array([z_on.index(z) + 1 if z in z_on else 0 for z in range(1, 31)], b.xref.dtype)
    b.abun = np.where(b.elem_on & (b.abun == 0), 1e-5, b.abun).astype(b.abun.dtype)
    ion = np.full((ion0.shape[0], len(z_on), ns), 1e-20)
    ion[:, :, 0] = 0.99999
    ion[:, :2, :3] = ion0[:, :2, :3]
    b.nElemUsed, b.nstages = len(z_on), ns
    return b, ion


# either side of the line between four cells to a wavefront and one (3
# channels), and the largest mesh: with the 16 rows and 16 channels that four
# cells side by side take at most, and with 32 rows
@pytest.mark.parametrize("nb,nSz,z_on,ns", [(410, 10, (1, 2), 7), (420, 10, (1, 2), 7), (4096, 16, (1, 2, 3, 4, 6), 9),
                                            (4096, 32, (1, 2), 7)])
def test_grains_on_large_meshes_match_oracle(nb, nSz, z_on, ns):
    print("grains on %d bins, %d sizes, elements" % (nb, nSz), z_on, flush=True)
    b, J, (Hden, Te0, Ne0, ion0), g, T0 = _on_mesh(nb, nSz)
    b, ion0 = _with_elements(b, ion0, z_on, ns)
    cells = np.arange(1, J.shape[0])[3::40]
    T = _context(J.shape[0] - 1, nb, b.nuArray)
    try:
        T.set_estimators(J)
        T.balance_setup(b)
        T.dust_setup(**_pe_tables(g))
        Tg, fl, nI, _, Te, Ne, ion = T.update_grains(T0, Hden=Hden, Te=Te0, Ne=Ne0, ionDen=ion0)
    finally:
        T.close()
    Teo, Neo, iono, flo, nIo, gdc, peh, _ = O.Balance(b).run_grains(J, Hden, Te0, Ne0, ion0, g, T0, "f64", cells=cells)
    To = O.dust_temps(J, T0, g, "f64", gdc=gdc, peh=peh)
    c = cells
    assert ((flo[c] & 16) == 0).sum() > len(c) // 2
    assert np.array_equal(fl[c], flo[c]) and np.array_equal(nI[c], nIo[c])
    assert np.max(np.abs(Te[c] - Teo[c]) / Teo[c]) < 1e-9
    assert np.max(np.abs(Ne[c] - Neo[c]) / Neo[c]) < 1e-9
    on = iono[c] > 0
    assert np.max(np.abs(ion[c][on] - iono[c][on]) / iono[c][on]) < 1e-8
    assert np.max(np.abs(Tg[c] - To[c]) / To[c].clip(1)) < 1e-9
