"""Host set-up of the exact coarse level: what it accepts and, where there is
no exact solve, why."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBDIR = os.path.join(ROOT, "stz_amd")


def test_verdicts(tmp_path):
    exe = str(tmp_path / "exact_level")
    subprocess.check_call(["g++", "-std=c++11", "-Wall", os.path.join(ROOT, "tests", "cpp", "exact_level.cc"),
                           "-o", exe, "-L", LIBDIR, "-lstz_amd", "-Wl,-rpath," + LIBDIR])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60, check=True).stdout.splitlines()
    assert out == ["solved", "0.125 0 0.0625", "is singular", "is not symmetric under reflection in x"]
