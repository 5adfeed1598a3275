"""The plans of the multi-iteration launches (lbm_amd/csrc/d2q9_plan.h),
checked on the host by tests/tile_plan_main.cpp: every node owned once, every
level's reads inside the level before it, every link once, every perimeter
slot one node, the launch limits.  CPU only."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tile_plans_cover_their_reads(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    exe = tmp_path / "tile_plan"
    cmd = [gxx, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
           os.path.join(ROOT, "tests", "tile_plan_main.cpp"), "-o", str(exe)]
    build = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr[-3000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, (run.returncode, run.stdout[-2000:], run.stderr[-2000:])
    assert run.stdout.startswith("ok "), run.stdout
