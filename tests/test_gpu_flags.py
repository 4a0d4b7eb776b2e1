"""Undefined bits of a context's flags mean nothing: the library keeps flags
of its own (crossing counts, viewing angles, far lattices) in the same word."""
import numpy as np
import pytest

from conftest import golden, oracle_problem
from mocassin_amd import _capi
from test_gpu_transport import transport_from_problem

pytestmark = pytest.mark.gpu


def test_undefined_flag_bits_are_ignored(monkeypatch):
    print("undefined flag bits", flush=True)
    g = golden("transport_c1mini_thick")
    out = []
    for extra in (0, 0x7fffffff & ~31):
        monkeypatch.setattr(_capi, "MC_GAS", 4 | extra)
        T = transport_from_problem(oracle_problem(g), int(g["seed"]))
        try:
            c = T.energy_packet_driver(1, 20000, 0)
            with pytest.raises(_capi.McError):
                T.crossings()                      # not enabled
            out.append((c,) + T.fetch())
        finally:
            T.close()
    (a, J, E), (b, K, F) = out
    assert all(a[k] == b[k] for k in ("n_seg", "n_abs", "n_esc", "n_lost", "n_line", "n_flights"))
    assert np.allclose(J, K, rtol=1e-10, atol=0) and np.allclose(E, F, rtol=1e-10, atol=0)
