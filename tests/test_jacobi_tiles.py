"""The plan of the vertex-tile Jacobi launches, run on the CPU
(tests/cpp/jacobi_tiles_check.cpp): what every tile reads, sums and passes on is
the plain iteration's, and every element and face is kept by one tile."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "xpbd-tissue-sim_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = tmp_path_factory.mktemp("jacobi_tiles") / "check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-pthread", "-I", CSRC, "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "cpp", "jacobi_tiles_check.cpp"), os.path.join(CSRC, "jacobi_tiles.cpp"),
                    os.path.join(CSRC, "mesh_tools.cpp"), "-o", str(exe)], check=True)
    return exe


# nx ny nz, instances, tiles (0: one an instance)
@pytest.mark.parametrize("case", ["1 1 1 1 1", "1 1 1 1 9", "6 5 7 1 0", "9 9 9 1 16", "12 12 12 1 256", "40 3 5 1 9",
                                  "4 6 3 5 6", "4 6 3 5 0", "4 6 3 5 60", "20 17 19 1 64", "3 3 3 1 1000"])
@pytest.mark.parametrize("late", [0, 1], ids=["contacts by patch", "contacts last"])
def test_tiles_give_the_plain_iteration(check, case, late):
    r = subprocess.run([str(check)] + case.split() + [str(late)], capture_output=True, text=True, timeout=60)
    print(case, "->", r.stdout.strip())
    assert r.returncode == 0, r.stdout + r.stderr
    if case.split()[4] == "0":   # an instance a tile: nothing runs twice
        assert "1.00 copies of an element, closed 1" in r.stdout
