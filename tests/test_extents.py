"""CPU check of tile counts near 2^31 elements along a dimension
(tests/c/extent_check.cpp, compiled here with g++ together with the planner
source)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tile_counts_of_extents_near_2_31(tmp_path):
    exe = str(tmp_path / "extent_check")
    src = [os.path.join(ROOT, "tests", "c", "extent_check.cpp"), os.path.join(ROOT, "ttc_amd", "csrc", "ttc_plan.cpp")]
    cmd = ["g++", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "include"),
           "-I" + os.path.join(ROOT, "ttc_amd", "csrc")] + src + ["-o", exe]
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if p.returncode != 0:
        pytest.fail("g++ failed:\n" + p.stdout)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    plans, lane, box, _ = [int(w) for w in r.stdout.replace(",", " ").split() if w.isdigit()][:4]
    assert plans > 20000 and lane > 300 and box > 10000, r.stdout
