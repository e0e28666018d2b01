"""CPU: the strips of elements that the strip kernels' threads take
(build_strips), on regular and irregular plans of one to many patches."""
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
    out = str(tmp_path_factory.mktemp("x") / "strip_check")
    subprocess.run([cxx, "-O1", "-std=c++17", f"-I{CSRC}", "-o", out,
                    os.path.join(ROOT, "tests", "cpp", "strip_check.cpp"),
                    os.path.join(CSRC, "mesh_plan.cpp")], check=True)
    return out


@pytest.mark.parametrize("shuffle", [False, True])
@pytest.mark.parametrize("dim,n,emax", [(2, 1, 768), (2, 9, 16), (2, 40, 100), (2, 60, 768), (3, 1, 768),
                                        (3, 4, 16), (3, 7, 33), (3, 12, 660), (3, 16, 660)])
def test_strips(exe, dim, n, emax, shuffle):
    r = subprocess.run([exe, str(dim), str(n), str(emax)] + ["shuffle"] * shuffle,
                       capture_output=True, text=True)
    print(r.stdout.strip())
    assert r.returncode == 0, r.stdout
