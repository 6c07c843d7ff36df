"""The engines' host code: when the HIP runtime fails, and what a prompt launches
(tests/cpp/engine_faults.cpp, built by __graft_entry__.build(): a C++ program
that puts its own runtime under the library, on the CPU)."""
import os
import subprocess

import pytest

from tests.conftest import ROOT

EXE = os.path.join(ROOT, "tests", "cpp", "engine_faults")


@pytest.mark.parametrize("what", ["launches", "memory", "folds"])
def test_engine_faults(what):
    assert os.path.exists(EXE), "tests/cpp/engine_faults is not built (run __graft_entry__.build())"
    r = subprocess.run([EXE, what], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
