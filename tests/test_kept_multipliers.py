"""Warm-started solves through the tile launches, with the host code's own launches
run tile by tile on the CPU (tests/cpp/kept_multipliers_check.cpp): a launch that
writes the solver-order multipliers must not be one that other tiles' copies read
them in."""
import subprocess

import pytest

from host_build import check_program

# solver, nx ny nz, instances, compute units -> the least number of tiles
CASES = [("gs 6 6 6 1 256", 1),       # an object a tile: nothing runs twice
         ("gs 4 6 3 5 256", 5),
         ("gs 12 10 9 1 256", 16),    # four lanes a cluster, four colours a launch
         ("gs 60 40 1 1 256", 16),    # one launch has all colours, and tiles that share clusters
         ("gs 24 22 23 1 64", 16),    # two colours a launch
         ("gs 22 24 23 1 16", 8),     # one lane a cluster, three colours
         ("gs 28 27 29 1 24", 8),     # two
         ("jacobi 5 5 5 1 256", 1),
         ("jacobi 4 4 3 5 256", 5),
         ("jacobi 12 10 9 1 256", 64),
         ("jacobi 14 9 11 3 256", 64)]


@pytest.mark.parametrize("case,tiles", CASES, ids=[c for c, _ in CASES])
def test_every_copy_starts_from_the_kept_multipliers(case, tiles):
    r = subprocess.run([check_program("kept_multipliers_check")] + case.split(), capture_output=True, text=True,
                       timeout=100)
    print(case, "->", r.stdout.strip())
    assert r.returncode == 0, r.stdout + r.stderr
    assert int(r.stdout.splitlines()[-1].split()[0]) >= tiles
