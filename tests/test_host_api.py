"""The entry points' host code without a device: the library linked to a program that
stands in for the HIP runtime (tests/hostapi/fake_hip.hpp), for allocation failures and
sizes that no GPU test should bring about."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

LIB = os.path.join(ROOT, "armsparse_amd")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = str(tmp_path_factory.mktemp("hostapi") / "host_api")
    src = os.path.join(ROOT, "tests", "hostapi")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-w", "-rdynamic", "-I", os.path.join(ROCM, "include"),
                    "-I", os.path.join(ROOT, "include"), os.path.join(src, "host_api.cpp"), "-o", exe,
                    "-L", LIB, "-larmsparse", f"-Wl,-rpath,{LIB}", f"-L{ROCM}/lib", "-lamdhip64",
                    f"-Wl,-rpath,{ROCM}/lib"], check=True, timeout=300)
    return exe


@pytest.mark.parametrize("check", ["no_memory", "launch_limits", "transpose_workspace", "narrow_batches",
                                   "vcsr_listing", "partitions", "max_launches"])
def test_host_code(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=300)
    print(r.stdout, r.stderr[-2000:])
    assert r.returncode == 0
