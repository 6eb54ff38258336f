"""Tables loaded into a session that holds fields already: the next solve's
rays take their emission and their absorption from the same tables."""
import numpy as np
import pytest

from oracle import oracle as O
from radchan_amd import VARIANT_BATCHED, VARIANT_PLAIN, Solver
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [False, True])
def test_reload(nb_tables, graph):
    """absorption coefficients that differ by a factor per table row; the
    band draws, which belong to the fields, are the same for both tables"""
    p, a, T = cases.nb_case(nb_tables, n=8, photmax=64)
    b = a.copy()
    b.kq[:] = a.kq * np.linspace(2.0, 0.25, a.nT, dtype=np.float32)[None, :, None]
    o = O.Oracle(p, b, T)
    de32, de32d, _, _ = o.solve(O.all_cells(p))
    o.close()
    s = Solver(p, a)
    s.set_fields([T])
    s.set_graph(graph)
    s.solve(VARIANT_BATCHED)
    s.load_tables(b)
    s.solve(VARIANT_BATCHED)
    assert np.abs(s.tallies() - de32d).max() <= 1e-12 * np.abs(de32d).max()
    s.solve(VARIANT_PLAIN)
    assert np.array_equal(s.tallies(), de32.astype(np.float64))
    s.close()
