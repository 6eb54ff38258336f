"""The walls' launch beside the fluid's: band keys sorted in registers and in
scratch (above 256 rays per cell), several solves in a row and a replayed
graph, against the oracle's FP64 sums of the FP32 tallies, from which the
batched ones differ only in order: 1e-12 of the largest."""
import numpy as np
import pytest

from oracle import oracle as O
from radchan_amd import VARIANT_BATCHED, Group, Solver
from tests import cases

pytestmark = pytest.mark.gpu


def _case(tables, photmax, mg):
    p, tab, T = cases.mg_case(tables, photmax=photmax) if mg else cases.nb_case(tables, photmax=photmax)
    p.calcwalls = 1
    return p, tab, T


def _tallies(s):
    return s.tallies(), s.surface()[2].reshape(-1, s.p.nVar)


def _want(p, tab, T):
    o = O.Oracle(p, tab, T)
    f, w = o.solve(O.all_cells(p))[1], o.solve(O.all_wall_cells(p), surface=True)[1]
    o.close()
    return f, w.reshape(-1, p.nVar)


def _close(a, b):
    for x, y in zip(a, b):
        assert np.abs(y).max() > 0
        assert np.abs(x - y).max() <= 1e-12 * np.abs(y).max()


@pytest.mark.parametrize("photmax", [64, 300])
@pytest.mark.parametrize("mg", [False, True])
def test_walls_beside_the_fluid(nb_tables, photmax, mg):
    p, tab, T = _case(nb_tables, photmax, mg)
    print(f"wall launch: {p.imax}x{p.jmax}x{p.kmax} photmax={photmax} levels={p.grid_num}", flush=True)
    s = Solver(p, tab)
    s.set_fields([T])
    want = _want(p, tab, T)
    for graph in (False, False, True, True):
        s.set_graph(graph)
        s.solve(VARIANT_BATCHED)
        _close(_tallies(s), want)
    s.close()


def test_group_walls_beside_the_fluid(nb_tables):
    p, tab, T = _case(nb_tables, 300, False)
    a, b = Solver(p, tab), Solver(p, tab)
    for s in (a, b):
        s.set_fields([T])
    want = _want(p, tab, T)
    g = Group([a, b])
    for _ in range(2):
        g.solve()
        _close(_tallies(a), want)
        _close(_tallies(b), want)
    g.close()
    a.close()
    b.close()
