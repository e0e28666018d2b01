"""CPU: which resident launches of several threads run together (resident_gate.h)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_admission(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no g++")
    exe = str(tmp_path / "gate_check")
    subprocess.run([cxx, "-O1", "-std=c++17", "-pthread",
                    "-I" + os.path.join(ROOT, "cudafemproject_amd", "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "gate_check.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
