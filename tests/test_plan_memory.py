"""Tile plans under host memory that runs out, on the CPU
(tests/cpp/plan_memory_check.cpp): meshes whose plans are built by one thread and by
several."""
import subprocess

import pytest

from host_build import check_program


@pytest.mark.parametrize("case", ["gs 9 9 9", "gs 60 22 22", "jacobi 9 9 9", "jacobi 16 16 16"])
def test_plans_survive_without_memory(case):
    r = subprocess.run([check_program("plan_memory_check")] + case.split(), capture_output=True, text=True, timeout=200)
    print(case, "->", r.stdout.strip())
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr[-300:])
