"""The re-emission tables on meshes whose bin count is no multiple of the four
bins that the ordered sums take at a time: the 200-bin deck without its last
bins, against the restatement with FP64 level populations."""
import copy

import numpy as np
import pytest

import mc_oracle as O
from conftest import balance_fixture, golden, grid_from_fixture
from mocassin_amd.atomic import emission_tables

pytestmark = pytest.mark.gpu


def _shortened(cut):
    """The c2mini deck's fixture and atomic bundle without its last bins."""
    g, b = golden("opacity_c2mini"), copy.copy(balance_fixture("c2mini")[0])
    nb = len(g["nuArray"]) - cut
    for k in ("nuArray", "widFlx", "em_gff", "em_gffHeII"):
        g[k] = g[k][:nb]
    for k in ("em_sHI", "em_sHeI", "em_sHeII"):
        g[k] = g[k][:len(g[k]) - cut]
    g["ints"] = g["ints"].copy()
    g["ints"][4] = nb
    nfb = int(g["em_ints"][9])
    m = g["em_fbm"][:4 * nfb].reshape(-1, 4).copy()
    rows = np.split(g["em_fbs"], np.cumsum(m[:, 3] - m[:, 2])[:-1])
    m[:, 3] = np.minimum(m[:, 3], nb)
    g["em_fbm"] = m.ravel()
    g["em_fbs"] = np.concatenate([r[:n] for r, n in zip(rows, m[:, 3] - m[:, 2])])
    b.nbins, b.nuArray = nb, b.nuArray[:nb]
    b.ch_sigma = np.ascontiguousarray(b.ch_sigma[:, :nb])
    b.ch_meta = b.ch_meta.copy()
    b.ch_meta[:, 4:7] = np.minimum(b.ch_meta[:, 4:7], nb)
    return g, b, nb


@pytest.mark.parametrize("cut", [1, 2, 3])
def test_tables_of_any_mesh_equal_oracle(cut):
    from mocassin_amd.transport import Transport
    g, b, nb = _shortened(cut)
    print("emission on %d bins" % nb, flush=True)
    axes, active, nc, _, fl, star_idx = grid_from_fixture(golden("opacity_c2mini"))
    T = Transport(*axes, active, nc, nb, b.nuArray, R_out=float(axes[0][-1]), geoCorr=(0, 0, 0),
                  ionEdge1=1.0, starPos=(0, 0, 0), starIdx=star_idx, deltaE=1.0, symmetric=fl["symmetric"], gas=True)
    ion = g["ionDen"].reshape(b.nstages, b.nElemUsed, nc + 1).transpose(2, 1, 0)
    try:
        T.balance_setup(b)
        T.emission_setup(**emission_tables(g))
        rec, tl, _ = T.emission_build(g["Hden"], g["Te"], g["Ne"], ion)
    finally:
        T.close()
    cells = np.arange(1, nc + 1)[::7]
    ex, tex = O.Balance(b).emission(O.emission_tables(g)[0], g["Te"], g["Ne"], ion, cells, "f64")
    # the bounds of the full mesh
    assert np.max(np.abs(rec[cells] - ex)) < 5e-7
    assert np.max(np.abs(tl[cells] / tex - 1)) < 2e-6
    assert np.all(rec[1:, -1] == 1.0)
