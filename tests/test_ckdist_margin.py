"""The margin around a bin's edges within which the correlated-k step forms
the exact power (radchan_amd/csrc/rc_ckbin.h), against the error of the quick
power with every FP32 rounding of it at its worst."""
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "radchan_amd", "csrc")


@pytest.fixture(scope="module")
def margin(tmp_path_factory):
    d = tmp_path_factory.mktemp("margin")
    (d / "t.cpp").write_text('#include <cstdio>\n#include <cstdlib>\n#include "rc_ckbin.h"\n'
                             "int main(int, char **v) { std::printf(\"%.17g\\n\", "
                             "rc::ck_edge_margin(std::atoi(v[1]), std::atof(v[2]))); }\n")
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(d / "t.cpp"), "-o", str(d / "t")], check=True)
    return lambda ie, pwr: float(subprocess.run([str(d / "t"), str(ie), repr(pwr)], capture_output=True, text=True,
                                                check=True).stdout)


def spread(n, seed):
    """k over the quick power's range, half of them near its ends"""
    rng = np.random.default_rng(seed)
    e = rng.uniform(-30.0, 30.0, n)
    e[: n // 4] = rng.uniform(27.0, 30.0, n // 4)
    e[n // 4: n // 2] = rng.uniform(-30.0, -27.0, n // 4)
    return 10.0 ** e


def ulps(x):
    """x in FP32 and its two neighbours"""
    x = x.astype(np.float32)
    return [x, np.nextafter(x, np.float32(np.inf)), np.nextafter(x, np.float32(-np.inf))]


@pytest.mark.parametrize("e", [1, 2, 3, 4, 5, 6, 7, 9, 10, 16, 33, 64])
def test_integer_law(margin, e):
    k, f = spread(40000, e), np.float32
    kf = k.astype(f)
    l0 = np.log2(kf.astype(np.float64))
    exact = np.exp(np.log(k.astype(np.longdouble)) / e)
    worst = 0.0
    for lg in ulps(l0):
        ok = np.abs(lg.astype(np.float64) - l0) <= np.spacing(np.abs(lg))
        y = f(1.0 / e) * lg
        for p0 in ulps(np.exp2(y.astype(np.float64))):
            p0 = p0.astype(np.float64)
            pe = np.prod(np.broadcast_to(p0, (e, len(k))), axis=0)
            for r in (1.0 - 2.0 ** -23, 1.0 + 2.0 ** -23):
                pk = p0 - p0 * ((pe - k) * (r / kf.astype(np.float64))) * (1.0 / e)
                worst = max(worst, float(np.abs((pk - exact) / exact)[ok].max()))
    assert margin(e, 1.0 / e) >= 10.0 * worst


@pytest.mark.parametrize("pwr", [0.02, 0.15, 0.7, 1.7, 7.0])
def test_other_laws(margin, pwr):
    """the logarithm corrected in FP64, its FP32 value an ulp off"""
    k = spread(40000, 3)
    exact = np.exp2(np.log2(k.astype(np.longdouble)) * np.longdouble(pwr))
    worst = 0.0
    for lg in ulps(np.log2(k.astype(np.float32).astype(np.float64))):
        l = lg.astype(np.float64)
        d = k * np.exp2(-l) - 1.0
        c = d * (d * (d / 3.0 - 0.5) + 1.0) * 1.4426950408889634
        worst = max(worst, float(np.abs((np.exp2(pwr * (l + c)) - exact) / exact).max()))
    assert margin(0, pwr) >= 10.0 * worst
