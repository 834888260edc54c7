"""The plan of the fused-colour Gauss-Seidel launches, run on the CPU
(tests/cpp/gs_tiles_check.cpp): what every tile reads, projects and passes on
gives the colour order's result exactly."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "xpbd-tissue-sim_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = tmp_path_factory.mktemp("gs_tiles") / "check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", CSRC, "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "cpp", "gs_tiles_check.cpp"), os.path.join(CSRC, "gs_tiles.cpp"),
                    os.path.join(CSRC, "mesh_tools.cpp"), "-o", str(exe)], check=True)
    return exe


# nx ny nz, instances, colours a launch, tiles (0: one an instance), clusters a block, waves
CASES = ["1 1 1 1 4 1 16 16", "6 5 7 1 8 0 16 16", "9 9 9 1 4 16 16 16", "9 9 9 1 2 16 64 8", "13 9 7 1 3 7 64 8",
         "40 3 5 1 4 9 16 3", "12 12 12 1 8 5 16 16", "4 6 3 5 4 6 16 16", "4 6 3 5 8 0 64 1", "20 17 19 1 2 64 64 2",
         "3 3 3 1 4 1000 16 16"]


@pytest.mark.parametrize("case", CASES)
def test_tiles_give_the_colour_order(check, case):
    r = subprocess.run([str(check)] + case.split(), capture_output=True, text=True, timeout=60)
    print(case, "->", r.stdout.strip())
    assert r.returncode == 0, r.stdout + r.stderr
    if case.split()[5] == "0":   # an instance a tile: nothing runs twice
        assert "1.00 copies, closed 1" in r.stdout
