"""Which launches the untuned Gauss-Seidel default makes, by size and iterations, on the
CPU (tests/cpp/tile_rule_check.cpp)."""
import subprocess

import pytest

from host_build import check_program


# a colour's clusters for each unit: 4, 49, 140 and 183
@pytest.mark.parametrize("case,least", [("6 6 6 8", 1), ("20 20 20 20", 1), ("22 22 23 10", 1), ("24 24 24 9", 2)])
def test_one_iteration_of_a_large_plan_runs_the_colours(case, least):
    for iters in (1, 2, 3):
        out = subprocess.run([check_program("tile_rule_check")] + case.split() + [str(iters)], check=True,
                             capture_output=True, text=True, timeout=60).stdout
        tiles, colours = (int(v) for v in out.split())
        assert (tiles > 0) == (iters >= least) and (colours > 0) == (iters < least), (iters, out)
