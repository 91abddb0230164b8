"""CPU replay of the one-tile-per-work-group row x column launch
(tests/c/lane_check.cpp, compiled here with g++ together with the planner
source): the work-group to tile map, every table and LDS index, each tile
element read and written exactly once with its true offsets, and out-of-range
offsets for every other slot."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_lane_launch_index_arithmetic(tmp_path):
    exe = str(tmp_path / "lane_check")
    src = [os.path.join(ROOT, "tests", "c", "lane_check.cpp"), os.path.join(ROOT, "ttc_amd", "csrc", "ttc_plan.cpp")]
    cmd = ["g++", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "include"),
           "-I" + os.path.join(ROOT, "ttc_amd", "csrc")] + src + ["-o", exe]
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if p.returncode != 0:
        pytest.fail("g++ failed:\n" + p.stdout)
    r = subprocess.run([exe, "60"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    walks, banded, full, tiles, partial, far = [int(w) for w in r.stdout.replace(",", " ").split() if w.isdigit()][:6]
    assert walks > 2000 and banded > 200 and full > 500 and partial > 1000 and tiles == 4 * walks and far == 2, r.stdout
