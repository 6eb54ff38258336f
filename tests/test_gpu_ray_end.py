"""Where a ray of the batched march ends: at a black wall whatever the
tolerance, after an optical depth that leaves nothing, and on absorption
coefficients that are no numbers, as in the plain march and the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from radchan_amd import VARIANT_BATCHED, VARIANT_PLAIN, Solver
from radchan_amd import fields as F
from radchan_amd import params as P

pytestmark = pytest.mark.gpu

TOLS = [1e-3, 1.7e-38, 1.6e-38, 1e-38, 1.5e-45]


def black_box(zbd, levels=None, maxs=None, photmax=100):
    """every face black: adiabatic x walls, fixed temperatures, or (zbd 4) the gas beside the z faces"""
    p = P.base_params(12, 6, 8, photmax=photmax, nVar=2, fact_mesh=1.5, seed=7, levels=levels, maxs=maxs)
    p.bd[:] = [2, 2, 2, 2, zbd, zbd]
    p.Tw[:] = [0.0, 0.0, 400.0, 420.0, 380.0, 390.0]
    p.calcwalls = 1
    return p


def check(p, tab, T):
    o = O.Oracle(p, tab, T)
    de32, de32d, _, _ = o.solve(O.all_cells(p))
    walls = o.solve(O.all_wall_cells(p), surface=True)[1].reshape(-1, p.nVar)
    o.close()
    s = Solver(p, tab)
    s.set_fields([T])
    s.solve(VARIANT_PLAIN)
    assert np.array_equal(s.tallies(), de32.astype(np.float64))
    s.solve(VARIANT_BATCHED)
    assert np.abs(s.tallies() - de32d).max() <= 1e-12 * np.abs(de32d).max()
    assert np.abs(s.surface()[2].reshape(-1, p.nVar) - walls).max() <= 1e-12 * np.abs(walls).max()
    s.close()


@pytest.mark.parametrize("tol", TOLS)
@pytest.mark.parametrize("zbd", [2, 4])
@pytest.mark.parametrize("levels", [False, True])
def test_tolerances(nb_tables, tol, zbd, levels):
    lv = dict(levels=[(12, 6, 8), (6, 3, 4)], maxs=[3, 400]) if levels else {}
    p = black_box(zbd, **lv)
    p.toll = p.tollS = tol
    check(p, nb_tables, F.channel_field(p, 500.0, 1500.0, noise=0.05, seed=3))


def test_opaque(nb_tables):
    """optical depths on both sides of 87, at which a step leaves nothing"""
    tab = nb_tables.copy()
    tab.kq[:] = tab.kq * (20.0 / np.median(tab.kq))
    p = black_box(2)
    p.toll = p.tollS = 1e-38
    check(p, tab, F.channel_field(p, 500.0, 1500.0, noise=0.05, seed=4))


def test_coefficients_that_are_no_numbers(nb_tables):
    """one cold cell whose table row holds NaN: what crosses it is NaN"""
    tab = nb_tables.copy()
    tab.kq[:, 0, :] = np.nan
    p = black_box(2, photmax=64)
    p.calcwalls = 0
    p.adiabw = p.adiabe = 0
    p.Tw[0] = p.Tw[1] = 460.0
    T = F.uniform_field(p, 1500.0, 1500.0).reshape(p.kmax + 2, p.jmax + 2, p.imax + 2)
    T[4, 3, 6] = float(tab.Tnb[0])
    T = T.reshape(-1)
    o = O.Oracle(p, tab, T)
    de32, de32d, _, _ = o.solve(O.all_cells(p))
    o.close()
    ok = ~np.isnan(de32d)
    assert 0 < ok.sum() < ok.size
    s = Solver(p, tab)
    s.set_fields([T])
    s.solve(VARIANT_PLAIN)
    assert np.array_equal(s.tallies(), de32.astype(np.float64), equal_nan=True)
    s.solve(VARIANT_BATCHED)
    b = s.tallies()
    s.close()
    assert np.array_equal(~np.isnan(b), ok)
    assert np.abs(b[ok] - de32d[ok]).max() <= 1e-12 * np.abs(de32d[ok]).max()
