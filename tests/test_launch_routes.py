"""Which tile a sparse GEMM call launches (tests/cpp/launch_routes.cpp, built by
__graft_entry__.build()), on the CPU."""
import os
import subprocess

from tests.conftest import ROOT

EXE = os.path.join(ROOT, "tests", "cpp", "launch_routes")


def test_gemm_routes():
    assert os.path.exists(EXE), "tests/cpp/launch_routes is not built (run __graft_entry__.build())"
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
