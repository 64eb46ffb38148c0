"""The wave's index loop (gpsm_amd/csrc/kernels/steps.h) at the ends of the
32-bit indices it runs over, on the CPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LAST = 2 ** 32 - 1  # the most entries an adjacency holds


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("steps") / "steps_driver")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "gpsm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "steps_driver.cpp"), "-o", exe], check=True)
    return exe


def test_steps_end_where_a_32_bit_index_wraps(driver):
    cases = [(0, 0), (0, 1), (0, 64), (0, 65), (7, 1031), (LAST // 1024 * 1024, LAST), (LAST - 1, LAST),
             (LAST - 63, LAST), (LAST - 64, LAST), (LAST - 255, LAST - 63)]
    p = subprocess.run([driver], input="".join("%d %d\n" % c for c in cases), capture_output=True, text=True,
                       check=True, timeout=60)
    for (lo, hi), line in zip(cases, p.stdout.split("\n")):
        want = range(lo, hi, 64)
        assert line.split() == ([str(len(want)), str(want[0]), str(want[-1]), "1"] if want else ["0", "0", "0", "1"])
