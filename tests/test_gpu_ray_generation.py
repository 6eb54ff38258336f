"""Ray generation of the batched kernel against the oracle, where its
lookups change form: the g CDF search by quarters (16 non-decreasing
entries) and the count over the row (other lengths, a row that decreases),
key / nQ by multiplication, band draws on the edges of the guide table, and
the radix sort's high digit of one bit up to eight."""
import numpy as np
import pytest

from oracle import oracle as O
from radchan_amd import VARIANT_BATCHED, VARIANT_PLAIN, Solver
from radchan_amd import fields as F
from radchan_amd import params as P
from radchan_amd.tables import Tables, synthetic_nb

pytestmark = pytest.mark.gpu


def cut_tables(nB, nQ, tab):
    """the first nQ g points of the first nB bands of `tab`, CDFs renormalised"""
    t = Tables(nB, tab.nT, nQ)
    for name in ("Tnb", "kP"):
        getattr(t, name)[:] = getattr(tab, name)
    for name in ("wvl", "wvr", "wvc", "kavg"):
        getattr(t, name)[:] = getattr(tab, name)[:nB]
    t.kq[:] = tab.kq[:nB, :, :nQ]
    t.prob[:] = tab.prob[:, :nB] / tab.prob[:, nB - 1:nB]
    t.probg[:] = tab.probg[:, :nB, :nQ] / tab.probg[:, :nB, nQ - 1:nQ]
    t.wq[:] = tab.wq[:nQ]
    return t


def solve_both(p, tab, T, estimator=0):
    s = Solver(p, tab)
    s.set_fields([T])
    o = O.Oracle(p, tab, T)
    de32, de32d, _, _ = o.solve(O.all_cells(p))
    s.solve(VARIANT_PLAIN)
    assert np.array_equal(s.tallies(), de32.astype(np.float64))
    s.solve(VARIANT_BATCHED)
    assert np.abs(s.tallies() - de32d).max() <= 1e-12 * np.abs(de32d).max()
    s.close()


@pytest.mark.parametrize("nB,nQ", [(5, 7), (37, 17), (360, 16), (3, 1), (16, 16), (17, 16), (360, 7)])
@pytest.mark.parametrize("photmax", [100, 300])
def test_table_shapes(nB, nQ, photmax):
    """nB nQ from 3 (no high digit) to 5760 keys, quarters and counts"""
    tab = cut_tables(nB, min(nQ, 16), synthetic_nb()) if nQ != 17 else cut17(nB)
    p = P.base_params(6, 4, 5, photmax=photmax, nVar=2, fact_mesh=1.5, seed=nB + nQ)
    p.nB, p.nQ = nB, nQ
    solve_both(p, tab, F.channel_field(p, 600.0, 1500.0, noise=0.02, seed=1))


def cut17(nB):
    """17 g points: the 16 of the synthetic tables and the last once more"""
    a = synthetic_nb()
    t = Tables(nB, a.nT, 17)
    for name in ("Tnb", "kP"):
        getattr(t, name)[:] = getattr(a, name)
    for name in ("wvl", "wvr", "wvc", "kavg"):
        getattr(t, name)[:] = getattr(a, name)[:nB]
    t.kq[:, :, :16], t.kq[:, :, 16] = a.kq[:nB], a.kq[:nB, :, 15]
    t.prob[:] = a.prob[:, :nB] / a.prob[:, nB - 1:nB]
    t.probg[:, :, :16], t.probg[:, :, 16] = 0.9 * a.probg[:, :nB], 1.0
    t.wq[:] = 1.0 / 17.0
    return t


@pytest.mark.parametrize("steps", [1, 64, 2048])
def test_guide_edges(steps):
    """band CDF values on multiples of 1/steps: draws equal to an entry and
    guide slots that hold none"""
    tab = synthetic_nb().copy()
    tab.prob[:] = np.ceil(tab.prob * steps) / steps
    p = P.base_params(4, 4, 4, photmax=200, nVar=2, fact_mesh=1.5, seed=steps)
    solve_both(p, tab, F.channel_field(p, 600.0, 1500.0, noise=0.02, seed=2))


@pytest.mark.parametrize("photmax", [100, 300])
@pytest.mark.parametrize("a,b", [(2, 3), (3, 4), (7, 8), (10, 12)])
def test_row_that_decreases(photmax, a, b):
    """g CDF rows of 16 with two entries exchanged: the count of entries up
    to R does not see their order, so the draws are those of the sorted rows;
    a search by quarters would find others"""
    tab = synthetic_nb()
    mixed = tab.copy()
    mixed.probg[:, ::5, a], mixed.probg[:, ::5, b] = tab.probg[:, ::5, b], tab.probg[:, ::5, a]
    p = P.base_params(6, 4, 5, photmax=photmax, nVar=2, fact_mesh=1.5, seed=a + b)
    T = F.channel_field(p, 600.0, 1500.0, noise=0.02, seed=4)
    o = O.Oracle(p, tab, T)
    de32, de32d, _, _ = o.solve(O.all_cells(p))
    o.close()
    s = Solver(p, mixed)
    s.set_fields([T])
    s.solve(VARIANT_PLAIN)
    assert np.array_equal(s.tallies(), de32.astype(np.float64))
    s.solve(VARIANT_BATCHED)
    assert np.abs(s.tallies() - de32d).max() <= 1e-12 * np.abs(de32d).max()
    s.close()


@pytest.mark.parametrize("nB", [513, 1024, 2000, 2048, 4095])
@pytest.mark.parametrize("photmax", [100, 257])
def test_high_digits(nB, photmax):
    """bands repeated up to nB: nB nQ of 8208 to 65520 keys, high digits of 6
    to 8 bits"""
    a = synthetic_nb()
    t = Tables(nB, a.nT, 16)
    pick = np.arange(nB) % a.nB
    for name in ("Tnb", "kP", "wq"):
        getattr(t, name)[:] = getattr(a, name)
    for name in ("wvl", "wvr", "wvc"):
        getattr(t, name)[:] = getattr(a, name)[pick]
    t.kavg[:] = np.random.default_rng(nB).permutation(nB) + 1.0
    t.kq[:] = a.kq[pick]
    t.prob[:] = ((np.arange(nB) + 1.0) / nB).astype(np.float32)
    t.probg[:] = a.probg[:, pick]
    p = P.base_params(6, 4, 5, photmax=photmax, nVar=2, fact_mesh=1.5, seed=nB)
    p.nB = nB
    solve_both(p, t, F.channel_field(p, 600.0, 1500.0, noise=0.02, seed=6))
