"""The shape of an autotuned handle's solves that the fused-colour launches do not run
(with attachments), from a cache file of the autotuner, on the CPU
(tests/cpp/tuned_shape_check.cpp; all its timings are equal, so the first shape wins)."""
import subprocess

import pytest

from host_build import check_program

QUAD, TILE = 4, 4000


def _shapes(path):
    out = subprocess.run([check_program("tuned_shape_check"), str(path)], check=True, capture_output=True, text=True,
                         timeout=60).stdout
    return [tuple(int(v) for v in line.split()) for line in out.splitlines()]


def test_the_autotuner_keeps_the_best_other_shape(tmp_path):
    path = tmp_path / "tune.txt"
    assert _shapes(path) == [(QUAD, TILE, 256), (QUAD, TILE, 64)]
    line = path.read_text().split()
    assert line[1:4] == ["4", "4000", "1"] and line[5] == "64"
    for plain in (128, -256):
        path.write_text(" ".join(line[:5] + [str(plain)]) + "\n")
        assert _shapes(path)[1] == (QUAD, TILE, plain)
    path.write_text(" ".join(line[:5]) + "\n")   # as they were before
    assert _shapes(path)[1] == (QUAD, TILE, 256)
    path.write_text(" ".join(line[:1] + ["4", "-1128", "1", "0.1"]) + "\n")
    assert _shapes(path)[1][:2] == (QUAD, -1128)


@pytest.mark.parametrize("plain", ["1064", "7", "4000"])
def test_a_shape_that_does_not_run_with_attachments_is_not_taken(tmp_path, plain):
    path = tmp_path / "tune.txt"
    _shapes(path)
    line = path.read_text().split()
    path.write_text(" ".join(line[:5] + [plain]) + "\n")
    assert _shapes(path)[1] == (QUAD, TILE, 64)   # tuned afresh
