"""The box walks' slab tests against the linear scan at scene scales from 2^-40
to 2^70, for the 4-wide nodes and their half-size form (tests/box_walk_check.cpp,
built with g++ from the library's host sources; CPU only)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_box_walks_match_the_scan_at_every_scale(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "box_walk_check")
    build = subprocess.run(
        ["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-I", os.path.join(ROOT, "include"),
         os.path.join(ROOT, "tests", "box_walk_check.cpp"),
         os.path.join(ROOT, "raydar_amd", "csrc", "bvh.cpp"), "-o", exe],
        capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-4000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert run.returncode == 0 and "box walks ok" in run.stdout, run.stdout + run.stderr
