"""The correlated-k kernel where it takes one way or another: bin laws with an
integer 1/pwr (bins from an FP32 power and one Newton step unless near an
edge) and without, values beyond the FP32 power's range, spectra so narrow
that every pair is near an edge, weights whose quotient leaves the normal
range, and sums of lengths around multiples of 16; against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from radchan_amd.spectra import ckdist

pytestmark = pytest.mark.gpu
GQ = (np.arange(16) + 0.5) / 16


def _check(spectra, dwv=0.01, **kw):
    off = np.concatenate([[0], np.cumsum([len(k) for k in spectra])])
    wv = np.concatenate([dwv * (1.0 + np.arange(len(k))) for k in spectra])
    wl = np.full(len(spectra), dwv)
    wr = np.array([dwv * max(len(k), 2) for k in spectra])
    print(f"ckdist paths: {[len(k) for k in spectra]} {kw}", flush=True)
    g = ckdist(off, wv, np.concatenate(spectra), wl, wr, GQ, **kw)
    kq, ka, lo, hi = O.ckdist(off, wv, np.concatenate(spectra), wl, wr, GQ, **kw)
    assert np.array_equal(g["kmin"], lo) and np.array_equal(g["kmax"], hi)
    np.testing.assert_allclose(g["kq"], kq, rtol=1e-12, atol=0)
    np.testing.assert_allclose(g["kavg"], ka, rtol=1e-12, atol=1e-300)


@pytest.mark.parametrize("pwr", [1.0, 0.5, 1.0 / 3.0, 0.125, 0.1, 1.0 / 64.0, 0.07, 2.0])
def test_bin_laws(pwr):
    rng = np.random.default_rng(int(1000 * pwr))
    _check([10.0 ** rng.uniform(-2.0, 3.0, 900), 10.0 ** rng.uniform(-8.0, 1.0, 700)], pwr=pwr)


@pytest.mark.parametrize("lo,hi", [(1e-28, 1e28), (1e-45, 1e-33), (1e33, 1e45), (1e-35, 1e-25), (2.0, 2.0 + 2e-9)])
def test_value_ranges(lo, hi):
    rng = np.random.default_rng(7)
    if hi / lo < 2.0:
        _check([rng.uniform(lo, hi, 600)])
    else:
        _check([np.exp(rng.uniform(np.log(lo), np.log(hi), 600))])


@pytest.mark.parametrize("dwv", [1e-120, 1e-90, 1e120])
def test_weights_beyond_the_reciprocal(dwv):
    _check([10.0 ** np.random.default_rng(3).uniform(-1.0, 2.0, 300)], dwv=dwv)


def test_sum_lengths():
    rng = np.random.default_rng(11)
    _check([10.0 ** rng.uniform(-1.0, 2.0, n) for n in (2, 3, 15, 16, 17, 18, 31, 33, 34, 49, 50, 257, 1001)])
