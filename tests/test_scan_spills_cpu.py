"""Registers that the first-pass scans spill, from the built library's kernel
descriptors: a few values parked outside the loop over the rows, not the lists'
or the accumulators' registers within it."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "simple-vector-db_amd", "libsvdb.so")
LLVM = "/opt/rocm/llvm/bin/"
MOST = 24  # of 256


@pytest.mark.skipif(not os.path.exists(LLVM + "llvm-readelf"), reason="no llvm-readelf")
def test_scans_keep_their_lists_in_registers(tmp_path):
    (tmp_path / "libsvdb.so").symlink_to(LIB)
    subprocess.run([LLVM + "llvm-objdump", "--offloading", "libsvdb.so"], cwd=tmp_path,
                   check=True, capture_output=True)
    spills = {}
    for f in sorted(tmp_path.glob("*gfx950*")):
        notes = subprocess.run([LLVM + "llvm-readelf", "--notes", str(f)], check=True,
                               capture_output=True, text=True).stdout
        for name, n in re.findall(r"\.symbol:\s+(\S+?)\.kd\b.*?\.vgpr_spill_count:\s+(\d+)", notes,
                                  re.S):
            spills[name] = int(n)
    scans = {k: v for k, v in spills.items() if "k_scan_bf16" in k or "k_scan_wide" in k}
    assert len(scans) > 100
    assert not {k: v for k, v in scans.items() if v > MOST}
