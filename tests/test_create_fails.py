"""Device memory that runs out at every allocation of a creation in turn, on the CPU
(tests/cpp/create_fails_check.cpp)."""
import subprocess

import pytest

from host_build import check_program


@pytest.mark.parametrize("case", ["gs 4 4 4", "gs 9 9 9", "jacobi 4 4 4", "jacobi 9 9 9"])
def test_nothing_is_left_of_a_handle_that_could_not_be_created(case):
    r = subprocess.run([check_program("create_fails_check")] + case.split(), capture_output=True, text=True, timeout=100)
    print(case, "->", r.stdout.strip())
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr[-300:])
