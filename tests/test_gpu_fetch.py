"""Results on their way to the host: table rows against the builds' own
column-major outputs, estimators of several pinned pieces, from two threads
at once, and the training data's checks, which run on the device."""
import ctypes as C
import threading

import numpy as np
import pytest

from mocassin_amd import _capi
from mocassin_amd._capi import McError

pytestmark = pytest.mark.gpu


def _lattice(n, nb):
    from mocassin_amd.transport import Transport
    nc = n ** 3 - 1
    act = np.zeros(n ** 3, np.int32)
    act[:nc] = np.random.default_rng(n).permutation(nc) + 1
    ax = np.linspace(0.0, 1.e17, n).astype(np.float32)
    return Transport(ax, ax, ax, act.reshape(n, n, n, order="F"), nc, nb, np.geomspace(1e-5, 25, nb).astype(np.float32),
                     R_out=1.e17, geoCorr=(0, 0, 0), ionEdge1=1.0, starPos=(0, 0, 0), starIdx=(1, 1, 1), deltaE=1.0)


# less than a piece, exactly two (4 MiB each: 2^20 doubles), and a ragged count
@pytest.mark.parametrize("n,nb", [(9, 65), (16, 256), (23, 130)])
def test_estimators_of_any_size_come_back_whole(n, nb):
    print("fetch", n, nb, flush=True)
    T = [_lattice(n, nb) for _ in range(2)]
    want = [np.random.default_rng(k).random((n ** 3, nb)) for k in range(2)]
    got = [[], []]
    try:
        for t, J in zip(T, want):
            J[0] = 0.0
            t.set_estimators(np.asfortranarray(J))

        def fetch(k):
            for _ in range(5):
                got[k].append(T[k].fetch()[0])
        th = [threading.Thread(target=fetch, args=(k,)) for k in range(2)]
        for t in th:
            t.start()
        for t in th:
            t.join()
    finally:
        for t in T:
            t.close()
    for k in range(2):
        assert len(got[k]) == 5 and all(np.array_equal(g, want[k]) for g in got[k])


# the smallest, columns of one brick, of several workgroups and on their edge (16
# points of 4 x 4 each 512 to a workgroup), ragged bricks, bins in slices
@pytest.mark.parametrize("shape,nb", [((2, 2, 2), 3), ((5, 3, 32), 7), ((4, 4, 33), 3), ((2, 9, 130), 31),
                                      ((13, 6, 27), 411), ((31, 30, 29), 61)])
def test_estimators_of_any_lattice_come_back(shape, nb):
    """Cells numbered in any order, a third of the positions inactive."""
    from mocassin_amd.transport import Transport
    print("lattice", shape, nb, flush=True)
    rng = np.random.default_rng(nb)
    n = int(np.prod(shape))
    nc = n - n // 3
    act = np.zeros(n, np.int32)
    act[rng.permutation(n)[:nc]] = rng.permutation(nc) + 1
    ax = [np.linspace(0.0, 1.e17, k).astype(np.float32) for k in shape]
    at = int(np.flatnonzero(act == 1)[0])
    star = np.unravel_index(at, shape, order="F")
    T = Transport(*ax, act.reshape(shape, order="F"), nc, nb, np.geomspace(1e-5, 25, nb).astype(np.float32), R_out=1.e17,
                  geoCorr=(0, 0, 0), ionEdge1=1.0, starPos=[float(a[k]) for a, k in zip(ax, star)],
                  starIdx=[int(k) + 1 for k in star], deltaE=1.0)
    try:
        want = rng.random((nc + 1, nb))
        want[0] = 0.0
        T.set_estimators(np.asfortranarray(want))
        assert np.array_equal(T.fetch()[0], want)
    finally:
        T.close()


@pytest.mark.parametrize("name", ["c2mini", "dust_pe"])
def test_table_rows_equal_the_columns(name):
    from test_gpu_emission import _ctx as emission_ctx
    from test_gpu_opacity import _ctx as opacity_ctx
    print("table rows", name, flush=True)
    for which, make in (("opacity", opacity_ctx), ("emission", emission_ctx)):
        T, g = make(name)[:2]
        try:
            nc1, nb, ns = T.nCells + 1, T.nbins, T._ns
            st = [np.ascontiguousarray(g[k], np.float32) for k in ("Hden", "Te", "Ne", "ionDen")]
            td = np.ascontiguousarray(g["Tdust"], np.float32) if name.startswith("dust") else None
            ptr = lambda a: None if a is None else a.ctypes.data
            cols = [np.full((nb, nc1), 7.0, np.float32) for _ in range(2)]
            rows = np.empty((nc1, nb), np.float32)
            with pytest.raises(McError, match="MC_ESTATE"):
                T._check(T._lib.mc_fetch_table_rows(T._h, 2 if which == "emission" else 0, rows.ctypes.data))
            with pytest.raises(McError, match="MC_EINVAL"):
                T._check(T._lib.mc_fetch_table_rows(T._h, 3, rows.ctypes.data))
            if which == "opacity":
                T._check(T._lib.mc_opacity_build(T._h, *map(ptr, st), ptr(td), ptr(cols[0]), ptr(cols[1]), None))
                for table, col in ((_capi.MC_TABLE_OPACITY, cols[0]), (_capi.MC_TABLE_SCATTERING, cols[1])):
                    assert np.array_equal(T._rows(table), col.T)
            else:
                T._check(T._lib.mc_emission_build(T._h, *map(ptr, st), ptr(td), ptr(cols[0]), None, None))
                assert np.array_equal(T._rows(_capi.MC_TABLE_RECPDF)[1:], cols[0].T[1:])
                assert np.all(cols[0][:, 0] == 7.0)            # row 0 is the caller's
        finally:
            T.close()


@pytest.mark.parametrize("bad", [("X", 5, np.nan), ("X", 72 * 300 - 1, np.inf), ("T", 40, -np.inf), ("M", 31, np.nan),
                                 ("M", 9299, -1.0)])
def test_training_data_is_checked(bad):
    from test_gpu_mlp import _ctx, _data, _random_net
    print("training data", bad, flush=True)
    D = dict(zip("XTM", _data(3, 300)))
    D[bad[0]].ravel()[bad[1]] = bad[2]
    D[bad[0]].ravel()[-1:] = bad[2]                           # the first is the one named
    T = _ctx()
    try:
        p, scale = _random_net(2)
        T.set_mlp(p, scale)
        for call in (lambda: T.mlp_loss_grad(D["X"], D["T"], D["M"]),
                     lambda: T.mlp_train(D["X"], D["T"], D["M"], np.arange(300), 300, 1e-3)):
            with pytest.raises(McError, match=r"MC_EINVAL.*entry %d not finite" % bad[1]):
                call()
        assert np.array_equal(T.get_mlp()[0], p.astype(np.float32))
    finally:
        T.close()
