"""What a batch of small objects and a large one takes of device memory, on the CPU
(tests/cpp/uneven_batch_check.cpp).  A plan needs a tile a unit, or as many as hold all
vertices in tiles as large as the largest object, whichever is more; objects that are
packed in turn leave at most half of each tile empty.  Against a batch of as many large
objects as units: twice the larger of one and the batches' vertices."""
import functools
import subprocess

import pytest

from host_build import check_program

# small cells, how many, large cells, units
CASES = ["1 3000 8 64", "2 200 8 24", "1 1000 5 16"]


@functools.lru_cache(maxsize=None)
def _held(case):
    r = subprocess.run([check_program("uneven_batch_check")] + case.split(), capture_output=True, text=True, timeout=100)
    print(case, "->", r.stdout.split("\n"))
    assert r.returncode == 0, r.stdout + r.stderr
    return [tuple(int(v) for v in line.split()) for line in r.stdout.splitlines()]


@pytest.mark.parametrize("case", CASES)
def test_plans_do_not_grow_with_the_number_of_small_objects(case):
    uneven, even = _held(case)
    assert uneven[2] == even[2] == 1   # an object (or several) a tile
    assert uneven[0] <= 2 * max(1, uneven[3] / even[3]) * even[0], (uneven, even)


@pytest.mark.parametrize("case", CASES)
def test_contacts_do_not_grow_with_the_number_of_small_objects(case):
    """A face has its records (under 200 bytes) and a place of 37 doubles and 4 int4 for a contact; the places of
    objects are alike within a factor of four."""
    small, count, large, units = (int(v) for v in case.split())
    faces = 12 * (count * small ** 2 + large ** 2)
    assert _held(case)[0][1] <= faces * (200 + 4 * (37 * 8 + 4 * 16))
