"""CPU check of the row copy's launch parameters (tests/c/row_check.cpp,
compiled here with g++ together with the planner source), up to the last
extents below 2^31."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_row_vectors_cover_each_row(tmp_path):
    exe = str(tmp_path / "row_check")
    src = [os.path.join(ROOT, "tests", "c", "row_check.cpp"), os.path.join(ROOT, "ttc_amd", "csrc", "ttc_plan.cpp")]
    cmd = ["g++", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "include"),
           "-I" + os.path.join(ROOT, "ttc_amd", "csrc")] + src + ["-o", exe]
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if p.returncode != 0:
        pytest.fail("g++ failed:\n" + p.stdout)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    plans, unaligned, last, small = [int(w) for w in r.stdout.replace(",", " ").split() if w.isdigit()][:4]
    assert plans > 5000 and unaligned > 1000 and last > 100 and small > 1000, r.stdout
