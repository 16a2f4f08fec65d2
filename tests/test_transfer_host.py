"""The staged copies between host arrays and the device (csrc/nuc_transfer.hip)
over a HIP runtime on the host: bytes, visibility of the staging memory, and
what a copy does to other threads and to its own.  Needs no GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANG = os.environ.get("ROCM_CLANG", "/opt/rocm/llvm/bin/clang++")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("transfer") / "test_transfer")
    subprocess.run([CLANG, "-x", "c++", "-O2", "-std=c++17", "-pthread", "-w",
                    "-I" + os.path.join(ROOT, "tests", "cpp", "host_hip"),
                    "-I" + os.path.join(ROOT, "nuc3d-cartisian_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_transfer.cpp"), "-o", exe], check=True, timeout=300)
    return exe


@pytest.mark.parametrize("case", ["bytes", "pinning", "locks", "device", "no_threads"])
def test_transfer(program, case):
    r = subprocess.run([program, case], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
