"""The opacity tables over lattices and cross-section sets where the division
of the bins changes: 4 to 16 wavefronts a tile, bins without entries, with one
to more than the 64 that a wavefront loads at a time, and cells of padding.
Against the sum in FP32 in segment order (bin 1 carries the free-free term
and is left out)."""
import numpy as np
import pytest

from conftest import balance_fixture

pytestmark = pytest.mark.gpu


def _lattice(n, b):
    from mocassin_amd.transport import Transport
    act = np.zeros(n ** 3, np.int32)
    at = np.random.default_rng(n).permutation(n ** 3)[:n ** 3 // 3]
    act[np.sort(at)] = np.arange(1, at.size + 1)
    ax = np.linspace(0.0, 1.e17, n).astype(np.float32)
    return Transport(ax, ax, ax, act.reshape(n, n, n, order="F"), at.size, b.nbins, b.nuArray, R_out=1.e17,
                     geoCorr=(0, 0, 0), ionEdge1=1.0, starPos=(0, 0, 0), starIdx=(1, 1, 1), deltaE=1.0)


# 8, 216, 512 and 1331 tiles; from no segment over most bins to 150 over some
@pytest.mark.parametrize("n,nseg,dense", [(5, 1, 1), (21, 40, 1), (30, 90, 60), (41, 12, 150)])
def test_tables_equal_the_ordered_sum(n, nseg, dense):
    b = balance_fixture("c2mini")[0]
    rng = np.random.default_rng(n)
    nb, on = b.nbins, [z for z in range(1, 31) if b.elem_on[z - 1]]
    segs, sigma = [], []
    for s in range(nseg + dense):
        z = int(rng.choice(on))
        ion = int(rng.integers(1, min(z, b.nstages) + 1))
        lo, hi = sorted(rng.integers(2, nb + 1, 2)) if s < nseg else (nb - 9, nb - 3)
        segs.append([z, ion, lo, hi])
        sigma.append((10.0 ** rng.uniform(-3, 0, hi - lo + 1)).astype(np.float32))
    T = _lattice(n, b)
    nc1 = T.nCells + 1
    Hden = rng.uniform(10, 1000, nc1).astype(np.float32)
    ion = (10.0 ** rng.uniform(-6, 0, (nc1, b.nElemUsed, b.nstages))).astype(np.float32)
    ion[rng.random(ion.shape) < 0.2] = 0.0                       # heavy ions that do not count
    print("opacity bins: %d tiles' lattice, %d segments" % (n, len(segs)), flush=True)
    try:
        T.balance_setup(b)
        T.opacity_setup(segs, np.concatenate(sigma), 1e-3)
        op = T.opacity_build(Hden, np.full(nc1, 9000.0, np.float32), Hden, ion)[0]
    finally:
        T.close()
    want = np.zeros((nc1, nb), np.float32)
    for (z, st, lo, hi), s in zip(segs, sigma):
        d = ion[:, int(b.xref[z - 1]) - 1, st - 1] * np.float32(b.abun[z - 1]) * Hden
        add = d if z <= 2 else np.where(d > 0, d, np.float32(0))
        want[:, lo - 1:hi] = want[:, lo - 1:hi] + s[None, :] * add[:, None]
    assert np.array_equal(op[1:, 1:].view(np.uint32), want[1:, 1:].view(np.uint32))
    assert np.all(op[0] == 0)
