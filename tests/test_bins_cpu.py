"""The 256-bin narrowing that the shortlist and the FP64 selection share
(svdb_bins.h) ends at the r-th smallest value, also for ranges that reach the
type's largest value — a C++ check on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_narrowing_ends_at_the_rth_value(tmp_path):
    exe = tmp_path / "bins_check"
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror",
                        "-I", os.path.join(ROOT, "simple-vector-db_amd", "csrc"),
                        "-o", str(exe), os.path.join(ROOT, "tests", "bins_check.cpp")],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
