"""Device functions run on the CPU as they stand in the HIP sources, 64 lanes in lockstep
(tests/wave/wave.hpp): arithmetic that inputs of a size, or with a fault, that no GPU
test should run would carry out of range."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

WAVE = os.path.join(ROOT, "tests", "wave")
HIP_INCLUDE = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("program", ["chunk_rows", "vcsr_medium", "max_gap", "max_bounds"])
def test_device_functions_stay_in_range(program, tmp_path):
    exe = str(tmp_path / program)
    # (the entry points of an included source are never called: their callees stay unresolved)
    subprocess.run(["g++", "-std=c++20", "-O1", "-g", "-w", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    "-I", HIP_INCLUDE, "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "armsparse_amd", "csrc"),
                    "-I", WAVE, os.path.join(WAVE, program + ".cpp"), "-Wl,--unresolved-symbols=ignore-all", "-o", exe],
                   check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout[-4000:], r.stderr[-4000:])
    assert r.returncode == 0
