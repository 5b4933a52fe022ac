"""Refused allocations (CPU only; tests/cpp/alloc_failure_test.cpp): the built
library's host code bound to a HIP of the test program's own, in which one
allocation after the other fails."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CPP = Path(__file__).resolve().parent / "cpp"


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("what", ["build", "truth"])
def test_refused_allocations(what):
    """build: a GPU build fails whichever allocation is refused, and frees nothing twice.  truth: ground truth runs
    without the memory of the matrix scan's lists."""
    subprocess.run(["make", "-C", str(CPP), "allocs"], check=True, capture_output=True, timeout=300)
    r = subprocess.run([str(CPP / "_build" / "alloc_failure_test"), what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
