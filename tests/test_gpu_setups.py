"""Several atomic set-ups on one context, each with other elements and stages:
the buffers that calls keep between them follow, one whose need grows while
another's shrinks among them.  Every call equals a fresh context's."""
import copy

import numpy as np
import pytest

from conftest import balance_fixture
from test_gpu_balance import _context
from test_gpu_balance_lanes import _subset
from test_gpu_mlp import _random_net

pytestmark = pytest.mark.gpu


def _decks():
    """(atomic data, cold state, lit state) of three element sets: 2 elements
    of 5 stages, 7 of 5 (38 REAL words a cell and 45 of the rows') and 4 of 9
    (39 and 43)."""
    b, J, Hden, Te0, Ne0, ion0, ref = balance_fixture("c2mini")
    for z_on, ns in (([1, 2], 5), ([1, 2, 6, 7, 8, 10, 16], 5), ([1, 2, 6, 7], 9)):
        sub, cold = _subset(b, ion0, z_on)
        lit = _subset(b, ref["ion"], z_on)[1]
        sub.nstages = ns
        wide = lambda a: np.concatenate([a, np.full(a.shape[:2] + (ns - 5,), 1e-20)], axis=2)
        yield sub, J.astype(np.float64), (Hden, Te0, Ne0, wide(cold)), (Hden, ref["Te"], ref["Ne"], wide(lit))


def _calls(T, b, J, cold, lit):
    T.balance_setup(b)
    T.set_estimators(J)
    out = list(T.line_luminosities(*lit)[:2])
    out += T.update_cells(*cold)[:5]
    return out + list(T.update_cells(*cold, warm_start=True, solver="secant", tol=1e-2)[:5])


def test_calls_after_another_set_up_equal_a_fresh_context():
    decks = list(_decks())
    nc, nb, nu = decks[0][1].shape[0] - 1, decks[0][0].nbins, decks[0][0].nuArray
    T = _context(nc, nb, nu)
    T.set_mlp(*_random_net(1))
    try:
        for b, J, cold, lit in decks + decks[::-1]:
            print("%d elements, %d stages" % (b.nElemUsed, b.nstages), flush=True)
            U = _context(nc, nb, nu)
            U.set_mlp(*_random_net(1))
            try:
                for x, y in zip(_calls(T, b, J, cold, lit), _calls(U, b, J, cold, lit)):
                    assert np.array_equal(x, y, equal_nan=True)
            finally:
                U.close()
    finally:
        T.close()
