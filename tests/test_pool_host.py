"""The pool of graph memory (gpsm_amd/csrc/pool.h) on the CPU, over a stub of
the HIP calls it makes: memory that waits goes back when an allocation of any
context, or outside the pools, fails; several threads at once."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pool(tmp_path):
    exe = str(tmp_path / "pool_driver")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "tests", "stub_hip"), "-I",
                    os.path.join(ROOT, "gpsm_amd", "csrc"), os.path.join(ROOT, "tests", "pool_driver.cpp"), "-o", exe],
                   check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert (p.returncode, p.stdout) == (0, "ok\n")
