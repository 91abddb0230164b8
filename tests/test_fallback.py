"""The planner's variants for pointers that are not aligned to a plan's vectors
(tests/c/fallback_check.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_variants_for_misaligned_pointers(tmp_path):
    exe = str(tmp_path / "fallback_check")
    src = [os.path.join(ROOT, "tests", "c", "fallback_check.cpp"), os.path.join(ROOT, "ttc_amd", "csrc", "ttc_plan.cpp")]
    cmd = ["g++", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "include"),
           "-I" + os.path.join(ROOT, "ttc_amd", "csrc")] + src + ["-o", exe]
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if p.returncode != 0:
        pytest.fail("g++ failed:\n" + p.stdout)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    own, moved, given = [int(w) for w in r.stdout.replace(",", " ").split() if w.isdigit()][:3]
    assert own > 1000 and moved > 30 and given > 500, r.stdout
