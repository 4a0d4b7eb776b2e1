"""Sweeps whose deposits go through the log (sorted and summed by range)
against the same sweeps with atomics: the same packets, so every counter is
equal and J and the escapes differ only in the order of FP64 sums."""
import numpy as np
import pytest

import mc_oracle as O
from conftest import golden, oracle_problem, view_from_fixture
from test_gpu_transport import transport_from_problem

pytestmark = pytest.mark.gpu

COUNTERS = ("n_seg", "n_abs", "n_sca", "n_esc", "n_lost", "n_line", "n_trapped", "n_flights")


def _sweep(T, kernel, n, first=0):
    T.set_tuning(kernel=kernel)
    T.zero_estimators()
    c = T.energy_packet_driver(1, n, first)
    return (c,) + T.fetch()


def _equal(a, b, n):
    """Two sums of the same k positive terms in different orders differ by at
    most 2 k 2^-53 of their value; a word gets a few terms a packet at most
    (the packets of these decks cross a cell once a flight)."""
    for k in COUNTERS:
        assert a[0][k] == b[0][k], k
    assert np.isclose(a[0]["qphot"], b[0]["qphot"], rtol=1e-9)
    rtol = 8.0 * n * 2.0 ** -53
    for x, y in zip(a[1:], b[1:]):
        assert np.array_equal(x > 0, y > 0)
        assert np.allclose(x, y, rtol=rtol, atol=0)


# packets: just above the log's smallest sweep, a ragged count, and one whose
# deposits (about 1e9) need more than one log: wavefronts save their packets
# and go on
@pytest.mark.parametrize("name,n", [("c1mini_thick", 400_001), ("full_mini_thick", 1_000_003), ("c3mini", 600_007),
                                    ("dust_mini_thick", 3_000_000), ("c3mini", 60_000_000)])
def test_logged_sweep_equals_atomics(name, n):
    g = golden("transport_" + name)
    print("log against atomics", name, n, flush=True)
    T = transport_from_problem(oracle_problem(g), int(g["seed"]))
    try:
        _equal(_sweep(T, "auto", n), _sweep(T, "one", n), n)
    finally:
        T.close()


@pytest.mark.parametrize("name", ["full_mini_view", "c1mini_view"])
def test_logged_viewing_angle_planes_equal_atomics(name):
    g = golden("transport_" + name)
    view = view_from_fixture(g)
    print("log against atomics, views", name, flush=True)
    T = transport_from_problem(oracle_problem(g, view=view), int(g["seed"]))
    try:
        T.set_view_angles(view)
        a, b = _sweep(T, "auto", 1_500_000, 2**32 - 5), _sweep(T, "one", 1_500_000, 2**32 - 5)
        assert a[2].shape[2] == 3
        _equal(a, b, 1_500_000)
    finally:
        T.close()


def test_contexts_share_the_log_and_crossing_counts_go_round_it():
    """A large sweep of one context, then one of another with fewer words;
    with crossing counts on the counts add up to the segments."""
    g, h = golden("transport_c3mini"), golden("transport_c1mini_thick")
    T, U = transport_from_problem(oracle_problem(g), 5), transport_from_problem(oracle_problem(h), 6)
    try:
        _equal(_sweep(T, "auto", 1_000_000), _sweep(T, "one", 1_000_000), 1_000_000)
        _equal(_sweep(U, "auto", 500_000), _sweep(U, "one", 500_000), 500_000)
        T.close()
        a = _sweep(U, "auto", 500_000)
        U.count_crossings(True)
        b = _sweep(U, "auto", 500_000)
        assert int(U.crossings().sum()) == int(b[0]["n_seg"])
        _equal(a, b, 500_000)
    finally:
        T.close()
        U.close()


@pytest.mark.parametrize("scale", [1e8, 1e10])
def test_far_lattice_equals_oracle(scale):
    """A lattice within 1e27 cm and one beyond it, whose wall distances take
    the general path: packet for packet the oracle's."""
    g = golden("transport_full_mini_thick")
    P0 = oracle_problem(g)
    s = np.float32(scale)
    P = O.Problem(xAxis=P0.xAxis * s, yAxis=P0.yAxis * s, zAxis=P0.zAxis * s, active=P0.active,
                  opacity=P0.opacity / s, nuArray=P0.nuArray, specCDF=P0.specCDF, R_out=P0.R_out * s,
                  geoCorr=np.asarray(P0.geoCorr, np.float32) * s, ionEdge1=P0.ionEdge1, deltaE=P0.deltaE,
                  starPos=P0.starPos, starIdx=P0.starIdx, recPDF=P0.recPDF, totalLines=P0.totalLines,
                  symmetric=P0.symmetric)
    print("far lattice", scale, float(np.abs(P.xAxis).max()), flush=True)
    T = transport_from_problem(P, 11)
    c = T.energy_packet_driver(1, 4000, 0)
    J, E = T.fetch()
    T.close()
    Jo, Eo, co = P.transport(0, 4000, 11, 1, O.MATH_OWN, O.J_FP64)
    for k in COUNTERS:
        assert c[k] == co[k], k
    assert np.allclose(J, Jo, rtol=1e-12, atol=0) and np.allclose(E, Eo, rtol=1e-12, atol=0)
