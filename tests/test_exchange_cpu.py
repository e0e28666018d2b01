"""CPU: the tables by which the workgroups of a resident solve exchange their
interface sums (build_exchange), on plans of one to many patches."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cudafemproject_amd", "csrc")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no g++")
    out = str(tmp_path_factory.mktemp("x") / "exchange_check")
    subprocess.run([cxx, "-O1", "-std=c++17", f"-I{CSRC}", "-o", out,
                    os.path.join(ROOT, "tests", "cpp", "exchange_check.cpp"),
                    os.path.join(CSRC, "mesh_plan.cpp")], check=True)
    return out


@pytest.mark.parametrize("dim,n,emax", [(2, 3, 768), (2, 9, 16), (2, 40, 100), (3, 2, 768),
                                        (3, 4, 16), (3, 7, 33), (3, 12, 768)])
def test_exchange_tables(exe, dim, n, emax):
    r = subprocess.run([exe, str(dim), str(n), str(emax)], capture_output=True, text=True)
    print(r.stdout.strip())
    assert r.returncode == 0, r.stdout
