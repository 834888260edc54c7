"""Handles without pinned memory, on the CPU (tests/cpp/no_pinned_check.cpp)."""
import subprocess

from host_build import check_program


def test_handles_do_without_pinned_memory():
    r = subprocess.run([check_program("no_pinned_check")], capture_output=True, text=True, timeout=60)
    print(r.stdout.strip())
    assert r.returncode == 0, r.stdout + r.stderr
