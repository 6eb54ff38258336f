"""How much scratch a solve takes where device memory is short
(radchan_amd/csrc/rc_scratch.h), on the host with a pretended memory."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "radchan_amd", "csrc")

HEAD = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include "rc_scratch.h"
static size_t left = 0;
struct Buf {
    size_t bytes = 0;
    int calls = 0;
    void release() { left += bytes; bytes = 0; }
    int ensure(size_t n) {
        if (n <= bytes) return 0;
        ++calls;
        release();
        if (n > left) return -11;
        left -= n;
        bytes = n;
        return 0;
    }
};
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
"""


def run(tmp_path, body, *args):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(HEAD + "int main(int argc, char **argv) {\n" + body + "\n    return 0;\n}\n")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=20)
    assert r.returncode == 0, r.stdout


# 64^3 cells of 100 rays, 2 runs: keys 50 MiB and tallies 200 MiB per run
FP64 = r"""
    const size_t rk = std::atoll(argv[1]), cells = 262144, P = 100, rr = cells * P, room = std::atoll(argv[2]);
    const int runs = std::atoi(argv[3]);
    left = room;
    Buf keys, ray;
    for (int again = 0; again < 3; ++again) {
        CHECK(rc::fp64_scratch(keys, ray, rk, rr, P, 2) == runs);
        if (!runs) continue;
        CHECK(keys.bytes >= rk * runs * 2);
        CHECK(ray.bytes >= P * 8 && ray.bytes <= ((size_t)1 << 28) * 8 && ray.bytes + keys.bytes + left == room);
        CHECK(ray.bytes / 8 >= P * runs && (runs == 1 || ray.bytes / 8 >= rr * runs));
    }
"""
K, R = 2 * 26214400, 8 * 26214400


@pytest.mark.parametrize("room,runs", [(2 * K + 2 * R, 2), (2 * K + 2 * R - 1, 1), (K + 2 * R, 1), (K + R, 1),
                                       (K + R // 2, 1), (K + 10000, 1), (K + 800, 1), (K + 799, 0), (K - 1, 0), (0, 0)])
def test_fp64_sorted(tmp_path, room, runs):
    """a solve runs wherever a run's keys and a unit's tallies fit"""
    run(tmp_path, FP64, 26214400, room, runs)


@pytest.mark.parametrize("room,runs", [(2 * R, 2), (2 * R - 1, 1), (800, 1), (799, 0)])
def test_fp64_unsorted(tmp_path, room, runs):
    run(tmp_path, FP64, 0, room, runs)


def test_fp64_keeps_to_2_GiB(tmp_path):
    run(tmp_path, r"""
    left = (size_t)1 << 40;
    Buf keys, ray;
    const size_t rr = (size_t)192 * 128 * 192 * 100;
    CHECK(rc::fp64_scratch(keys, ray, rr, rr, 100, 2) == 1);
    CHECK(ray.bytes == (size_t)1 << 31 && keys.bytes == rr * 2);
    const int calls = keys.calls + ray.calls;
    CHECK(rc::fp64_scratch(keys, ray, rr, rr, 100, 2) == 1 && keys.calls + ray.calls == calls);
""")


SORT = r"""
    left = std::atoll(argv[3]);
    const size_t fluid = std::atoll(argv[1]), walls = std::atoll(argv[2]);
    const int want = std::atoi(argv[4]);
    Buf b;
    size_t refused = 0;
    for (int again = 0; again < 3; ++again) {
        const int calls = b.calls;
        CHECK(rc::sort_scratch(b, fluid, walls, refused) == want);
        if (want >= 0) CHECK(b.bytes >= 2 * (want ? fluid + walls : fluid > walls ? fluid : walls));
        if (want >= 0 && again) CHECK(b.calls == calls);
    }
"""


@pytest.mark.parametrize("fluid,walls,room,want", [(1000, 300, 2600, 1), (1000, 300, 2599, 0), (1000, 300, 2000, 0),
                                                   (300, 1000, 2000, 0), (1000, 300, 1999, -1), (1000, 0, 2000, 1),
                                                   (1000, 0, 1999, -1), (0, 0, 0, 1)])
def test_sort_scratch(tmp_path, fluid, walls, room, want):
    """the walls' keys beside the fluid's, else in their place"""
    run(tmp_path, SORT, fluid, walls, room, want)


def test_sort_scratch_grows(tmp_path):
    """other schedules of one session: a smaller pair of sizes is tried again"""
    run(tmp_path, r"""
    left = 2000;
    Buf b;
    size_t refused = 0;
    CHECK(rc::sort_scratch(b, 900, 300, refused) == 0 && refused == 2400);
    CHECK(rc::sort_scratch(b, 600, 200, refused) == 1);
    CHECK(rc::sort_scratch(b, 700, 250, refused) == 1 && b.bytes == 1900);
    CHECK(rc::sort_scratch(b, 900, 300, refused) == 0 && b.bytes == 1900);
""")
