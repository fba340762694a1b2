"""Vector registers of kernels whose speed is the number of waves that a SIMD holds, read
from the metadata of the library as built: 64 registers leave 8 waves of 64 lanes, 72
leave 7."""
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


@pytest.fixture(scope="module")
def vgprs(tmp_path_factory):
    """{demangled kernel name up to its arguments: VGPRs}"""
    tools = [shutil.which(t, path=LLVM + os.pathsep + os.environ["PATH"]) for t in ("llvm-objdump", "llvm-readelf", "c++filt")]
    if None in tools:
        pytest.skip("needs llvm-objdump, llvm-readelf and c++filt")
    d = str(tmp_path_factory.mktemp("objects"))
    shutil.copy(os.path.join(ROOT, "armsparse_amd", "libarmsparse.so"), d)
    subprocess.run([tools[0], "--offloading", "libarmsparse.so"], cwd=d, check=True, capture_output=True, timeout=120)
    found = {}
    for f in sorted(os.listdir(d)):
        if not f.endswith("gfx950"):
            continue
        notes = subprocess.run([tools[1], "--notes", f], cwd=d, check=True, capture_output=True, text=True, timeout=120).stdout
        pairs = re.findall(r"\.symbol:\s+(\S+)\.kd.*?\.vgpr_count:\s+(\d+)", notes, re.S)
        names = subprocess.run([tools[2]], input="\n".join(n for n, _ in pairs), check=True, capture_output=True, text=True,
                               timeout=120).stdout.split("\n")
        for name, (_, n) in zip(names, pairs):
            found[re.sub(r"\(anonymous namespace\)::|armsp::|^void ", "", name).split("(")[0]] = int(n)
    return found


@pytest.mark.parametrize("coo", ["true", "false"])
@pytest.mark.parametrize("kernel,most", [("unsigned short, 8, 8", 64), ("unsigned short, 4, 8", 64), ("float, 4, 4", 64),
                                         ("float, 8, 4", 72)])
def test_sddmm_without_column_halves(vgprs, kernel, most, coo):
    assert vgprs[f"k_sddmm_stream<{kernel}, {coo}, true>"] <= most
