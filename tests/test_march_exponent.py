"""The march's exponentials (radchan_amd/csrc/rc_expm1.h) on the host: the
bulk march's form gives what the plain march's gives, and ends a ray at a
black wall whatever the tolerance."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "radchan_amd", "csrc")

SRC = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <limits>
#include "rc_expm1.h"
static uint32_t bits(float f) { uint32_t u; std::memcpy(&u, &f, 4); return u; }
static float value(uint32_t u) { float f; std::memcpy(&f, &u, 4); return f; }
static bool same(float a, float b) { return bits(a) == bits(b) || (a != a && b != b); }
static long bad = 0;
static void check(float d) {
    float m0, e0, m1, e1;
    rcd::expm1_exp_le88(-d, m0, e0);
    rcd::expm1_exp_step(d, false, m1, e1);
    if (!same(e0, e1) || !(same(m0, m1) || (m0 == 0.f && m1 == 0.f))) {
        if (!bad++) std::printf("depth %a: expm1 %a %a, exp %a %a\n", d, m0, m1, e0, e1);
    }
    rcd::expm1_exp_step(d, true, m1, e1);
    if (bits(e1) != 0u || m1 != -1.0f) {
        if (!bad++) std::printf("wall, depth %a: expm1 %a, exp %a\n", d, m1, e1);
    }
}
int main() {
    for (uint32_t u = bits(80.f); u <= bits(110.f); u += 7) check(value(u));
    for (uint32_t u = 0; u < 0x7F800000u; u += 65521) check(value(u));
    const float inf = std::numeric_limits<float>::infinity();
    for (float d : {0.f, -0.f, 87.f, std::nextafter(87.f, 0.f), std::nextafter(87.f, inf), 87.68f, 88.03f, inf,
                    std::numeric_limits<float>::quiet_NaN(), -1e-6f})
        check(d);
    return bad ? 1 : 0;
}
"""


@pytest.mark.parametrize("opt", ["-O0", "-O2"])
def test_step_form(tmp_path, opt):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", opt, "-ffp-contract=off", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
