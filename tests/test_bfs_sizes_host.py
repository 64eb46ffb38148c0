"""The breadth-first join's level buffers (gpsm_amd/csrc/host/bfs_sizes.h) on
the CPU: their layout, the bound on the first request, and what is asked for
next where the device has no room."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GB = 1 << 30
LEAST, MOST = 1 << 18, 1 << 24


@pytest.fixture(scope="module")
def sizes(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("bfs") / "bfs_sizes_driver")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "gpsm_amd", "csrc", "host"),
                    os.path.join(ROOT, "tests", "bfs_sizes_driver.cpp"), "-o", exe], check=True)

    def run(*case):
        out = subprocess.run([exe], input=" ".join(map(str, case)) + "\n", capture_output=True, text=True, check=True,
                             timeout=60).stdout
        head, tail = out.split("|")
        head = [int(x) for x in head.split()]
        lv = [int(x) for x in tail.split()]
        return bool(head[0]), head[2:], [lv[i:i + 4] for i in range(0, len(lv), 4)]

    return run


@pytest.mark.parametrize("widest", [3, 4, 5, 8])
@pytest.mark.parametrize("first", [1, 12345, 1 << 25])
@pytest.mark.parametrize("expected", [0.0, 5e4, 1e12])
def test_layout_and_bound(sizes, widest, first, expected):
    slack = 8192 * 64
    ok, asked, levels = sizes(widest, first, slack, expected, 16.0 * GB, 1 << 60)
    assert ok and len(asked) == 1 and len(levels) == widest - 2
    rows = min(max(16 * int(expected), LEAST), MOST)
    end = 0
    for i, (at, cap, long_cap, words) in enumerate(levels):
        level = i + 1
        assert at == end and words >= 6 + level + 1 and words % 2 == 0
        assert cap == slack + (first if level == 1 else rows)
        assert long_cap == (first if level == 1 else cap // 16)
        end = at + (cap + long_cap) * words
    assert asked[0] == 4 * end <= 16 * GB * 4 // 5


def test_less_room_halves_the_rows(sizes):
    case = (6, 1 << 20, 8192 * 64, 1e9, 16.0 * GB)
    full = sizes(*case, 1 << 60)[1][0]
    least = None
    for room in (full * 5 // 4, full, full // 2, full // 8, full // 16):
        ok, asked, levels = sizes(*case, room)
        assert asked[0] == full and all(a > b for a, b in zip(asked, asked[1:]))
        assert asked[-1] * 5 // 4 <= room if ok else levels[1][1] == 8192 * 64 + LEAST
        assert levels[0][1] == (1 << 20) + 8192 * 64  # level 1 is always whole
        least = asked[-1]
    ok, asked, levels = sizes(*case, least // 2)
    assert not ok and levels[1][1] == 8192 * 64 + LEAST


def test_a_small_bound_holds_level_one(sizes):
    """Rows shrink to their least where the bound leaves no more."""
    ok, asked, levels = sizes(8, 1 << 25, 8192 * 64, 1e12, 4.0 * GB, 1 << 60)
    assert ok and LEAST <= levels[1][1] - 8192 * 64 < MOST
    assert asked[0] * 5 // 4 <= 4 * GB
    assert sizes(8, 1 << 25, 8192 * 64, 1e12, 1.0 * GB, 1 << 60)[2][1][1] == 8192 * 64 + LEAST
