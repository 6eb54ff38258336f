"""The spline restriction's kernels at the line lengths where they change
form (64, 32, 16, 8, 4 and 2 lines per workgroup, and lines beyond LDS), along
each axis, and on values outside the range its quotients by reciprocals
cover: equal to the oracle bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O
from radchan_amd import params as P
from radchan_amd.solver import spline_restrict

pytestmark = pytest.mark.gpu


def _check(n, coarse, T, seed=0):
    p = P.base_params(*n, photmax=8, nVar=1, fact_mesh=1.5, seed=seed, levels=[n, coarse], maxs=[4, 64])
    print(f"spline lines: {n} -> {coarse}", flush=True)
    tc, tw = spline_restrict(p, 1, T)
    oc, ow = O.interp3d(p, 1, T)
    for got, want in ((tc, oc.astype(np.float32)), (tw, ow.astype(np.float32))):
        nan = np.isnan(want)                 # overflowed lines: a NaN's sign and payload are not defined
        assert np.array_equal(np.isnan(got), nan)
        assert np.array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])


def _field(n, seed):
    rng = np.random.default_rng(seed)
    return (900.0 + 300.0 * rng.standard_normal((n[2] + 2, n[1] + 2, n[0] + 2)).clip(-2.5, 2.5)).astype(np.float32)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("n,r", [(2, 1), (2, 2), (6, 3), (8, 2), (12, 4), (104, 2), (106, 2), (208, 2), (210, 5),
                                 (404, 4), (406, 2), (766, 2), (768, 3), (1380, 2), (1382, 2), (2456, 2), (2458, 2)])
def test_line_lengths(axis, n, r):
    size = [4, 6, 10]
    size[axis] = n
    coarse = [2, 3, 5]
    coarse[axis] = n // r
    _check(tuple(size), tuple(coarse), _field(size, n + axis))


@pytest.mark.parametrize("what", ["tiny", "huge", "both", "edge"])
def test_values_beyond_the_reciprocals(what):
    n = (16, 12, 70)
    T = _field(n, 3)
    if what == "tiny":
        T *= np.float32(1e-36)
    elif what == "huge":
        T *= np.float32(1e34)
    elif what == "both":
        T[20:30] *= np.float32(1e-30)
        T[40:] *= np.float32(1e30)
    else:
        T[::7] = np.float32(1e-15)
        T[3::7] = np.float32(1e15)
    with np.errstate(over="ignore", invalid="ignore"):
        _check(n, (8, 6, 35), T)
