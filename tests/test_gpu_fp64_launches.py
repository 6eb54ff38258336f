"""The FP64 variant where its launches are split: fields whose ray tallies
exceed the scratch of one launch (2^28 rays), by cells and by runs, and
fields of few rays per cell: equal to the oracle's FP64 sums bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O
from radchan_amd import VARIANT_PLAIN, Solver
from tests import cases

pytestmark = pytest.mark.gpu


def _check(p, tab, T, cells):
    p.fp64 = 1
    print(f"fp64 launches: {p.imax}x{p.jmax}x{p.kmax} photmax={p.photmax} nVar={p.nVar}", flush=True)
    s = Solver(p, tab)
    s.set_fields([T])
    st = s.solve(VARIANT_PLAIN)
    got = s.tallies()
    o = O.Oracle(p, tab, T)
    every = O.all_cells(p)
    _, want, _, steps = o.solve([every[c] for c in cells], precision=1)
    assert np.array_equal(got[cells], want)
    assert st["rays"] == len(every) * p.photmax * p.nVar
    if len(cells) == len(every):
        assert st["steps"] == steps.sum()
    s.close()
    o.close()


@pytest.mark.parametrize("photmax,nVar", [((1 << 19) + 5, 2),      # 511 cells, then 1
                                          (200000, 3)])            # two runs, then one
def test_split_launches(photmax, nVar):
    p, tab, T = cases.grey_case(n=8)
    p.photmax, p.nVar = photmax, nVar
    _check(p, tab, T, [0, 511])


@pytest.mark.parametrize("photmax", [1, 3, 65])
def test_few_rays(nb_tables, photmax):
    p, tab, T = cases.nb_case(nb_tables, photmax=photmax)
    _check(p, tab, T, list(range(p.imax * p.jmax * p.kmax)))
