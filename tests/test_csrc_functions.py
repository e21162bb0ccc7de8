"""The host-callable functions that the kernels and their host code are made of, checked as they are:
csrc_checks.cpp is built against the library's headers and its shared library, and each of its checks
is one test."""
import os
import subprocess
from pathlib import Path

import pytest

import ocfd_amd as A

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "opencfd-ec_amd" / "csrc"


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = tmp_path_factory.mktemp("csrc") / "checks"
    lib = Path(A.LIB_PATH)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-Wno-unused-result", f"-I{CSRC}",
                    str(HERE / "csrc_checks.cpp"), "-x", "none", str(lib), f"-Wl,-rpath,{lib.parent}", "-o", str(out)], check=True)
    return str(out)


@pytest.mark.parametrize("check", ["give_up", "vector_groups", "face_tiles", "sweep_tables"])
def test_check(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
