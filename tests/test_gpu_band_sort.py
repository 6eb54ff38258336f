"""The band keys' sort in registers (up to 128 and up to 256 rays) and past it:
FP64 sums in the keys' order, fluid and walls, equal to the oracle's bit for
bit."""
import numpy as np
import pytest

from oracle import oracle as O
from radchan_amd import VARIANT_PLAIN, Solver
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("photmax", [1, 2, 63, 64, 65, 127, 128, 129, 191, 255, 256, 257])
def test_sorted_keys(nb_tables, photmax):
    p, tab, T = cases.nb_case(nb_tables, n=8, photmax=photmax)
    p.fp64 = p.calcwalls = 1
    print(f"band sort: photmax={photmax}", flush=True)
    s = Solver(p, tab)
    s.set_fields([T])
    s.solve(VARIANT_PLAIN)
    o = O.Oracle(p, tab, T)
    assert np.array_equal(s.tallies(), o.solve(O.all_cells(p), precision=1)[1])
    walls = o.solve(O.all_wall_cells(p), surface=True, precision=1)[1]
    assert np.array_equal(s.surface()[2].reshape(-1, p.nVar), walls.reshape(-1, p.nVar))
    s.close()
    o.close()
