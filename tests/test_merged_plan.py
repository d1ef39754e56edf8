"""The merged solves' plan (psp_amd/csrc/symbolic.cpp: BuildMerged,
DefaultSlices, BuildBlockTiles) checked on the host by
tests/merged_plan_check.cpp, built here with the address and undefined
sanitizers: both solve passes emulated from the tiles, block lists and vector
rows against the fine elimination tree, every index against its array, and
the fold's lists writing every factor entry once.  Small, ragged and flat
grids, single points of a side, leaves of one point and of 48, both factor
precisions, one to many inner slices per tile."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("merged") / "merged_plan_check")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "psp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "merged_plan_check.cpp"),
                    os.path.join(ROOT, "psp_amd", "csrc", "symbolic.cpp"), "-o", exe], check=True)
    return exe


# nx ny nz [precision cutoff minTiles maxSplit slice]
@pytest.mark.parametrize("args", [
    "24 20 26", "9 13 27 1", "12 10 24", "3 3 22", "13 1 24", "16 16 20 0 1", "30 20 26 0 5 1 1",
    "40 40 24 1", "40 40 24 0 12 4096 16", "26 22 24 0 12 256 8 3", "64 20 22 1 48", "61 47 30",
])
def test_merged_plan(checker, args):
    out = subprocess.run([checker] + args.split(), capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, (out.stdout + out.stderr)[-3000:]
    assert "class 0:" in out.stdout
