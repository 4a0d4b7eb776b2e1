"""The network's input rows on meshes whose bin count is no multiple of the 16
bins that the integrals take at a time: the bands of one cell end in its own
row, whatever the mesh.  Every lattice point is a cell, so that each row has
a neighbour."""
import copy

import numpy as np
import pytest

from conftest import balance_fixture
from mocassin_amd import mlp as MP

pytestmark = pytest.mark.gpu


# the least mesh, meshes with several band ends to a bin of the last step
# beyond the mesh (65 to 113), multiples of 16 and their neighbours
@pytest.mark.parametrize("nb", [64, 65, 71, 72, 80, 81, 83, 85, 96, 97, 98, 99, 112, 113, 114, 130, 199])
def test_features_of_any_mesh_match_their_definition(nb):
    from mocassin_amd.transport import Transport
    print("mlp features on %d bins" % nb, flush=True)
    b = copy.copy(balance_fixture("c2mini")[0])
    b.nbins, b.nuArray = nb, np.ascontiguousarray(b.nuArray[:nb])
    b.ch_sigma = np.ascontiguousarray(b.ch_sigma[:, :nb])
    b.ch_meta = b.ch_meta.copy()
    b.ch_meta[:, 4:7] = np.minimum(b.ch_meta[:, 4:7], nb)
    n, nc = 5, 125
    rng = np.random.default_rng(nb)
    J = rng.uniform(0.1, 10.0, (nc + 1, nb)) * 10.0 ** rng.uniform(-8, 2, (nc + 1, 1))
    J[::11] = 0.0
    Hden = 10.0 ** rng.uniform(1, 4, nc + 1)
    ax = np.linspace(0.0, 1.e17, n).astype(np.float32)
    T = Transport(ax, ax, ax, np.arange(1, nc + 1, dtype=np.int32).reshape(n, n, n, order="F"), nc, nb, b.nuArray,
                  R_out=1.e17, geoCorr=(0, 0, 0), ionEdge1=1.0, starPos=(0, 0, 0), starIdx=(1, 1, 1), deltaE=1.0)
    try:
        T.balance_setup(b)
        T.set_estimators(J)
        X, hit = T.mlp_features(Hden, jscale=2.0)
    finally:
        T.close()
    # FP32 logarithms, at most 30: an ulp of those
    bound = 4e-6
    edge = [i * nb // 64 for i in range(65)]
    bands = np.stack([2.0 * J[1:, edge[i]:edge[i + 1]].sum(axis=1) for i in range(64)], axis=1)
    assert np.array_equal(hit[1:].astype(bool), J[1:].max(axis=1) > 0)
    assert np.max(np.abs(X[:, :64] - np.log10(np.maximum(bands, 1e-30)))) < bound
    assert np.max(np.abs(X[:, 64] - np.log10(Hden[1:]))) < bound
    for k, z in enumerate(MP.SLOTS_Z):
        assert np.max(np.abs(X[:, 65 + k] - (np.log10(b.abun[z - 1]) if b.elem_on[z - 1] else -30.0))) < bound
