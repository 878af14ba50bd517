"""The partial lists of the FP64 scan (svdb_f64_lists.h): within the limits that a
search was ever accepted with, large enough for a cut to make room, and small
for a small k — a C++ check on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_lists_fit_and_can_be_cut(tmp_path):
    exe = tmp_path / "f64_lists_check"
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror",
                        "-I", os.path.join(ROOT, "simple-vector-db_amd", "csrc"),
                        "-o", str(exe), os.path.join(ROOT, "tests", "f64_lists_check.cpp")],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
