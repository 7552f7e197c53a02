"""CPU test of the host-side launch planning (csrc/host_plan.h): the C++ unit
test in tests/cpp_host is compiled with g++ (no HIP) and run.  It covers the
partials a decode launch leaves to its consumer for 1 to 16 rows, with guard
words around the plan, and the tokens of one launch of an append, whose threads
stay below a launch's limit."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_host_plan(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "test_host_plan"
    cmd = [gxx, "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{ROOT / 'streaming-attention_amd' / 'csrc'}",
           str(ROOT / "tests" / "cpp_host" / "test_host_plan.cpp"), "-o", str(exe)]
    subprocess.run(cmd, check=True, capture_output=True, text=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr
    assert "all checks passed" in res.stdout
