"""The bf16 copy of a matrix with its column sums, in one pass or, without workspace, in two."""
import os
import subprocess
import sys

import pytest
import torch

from conftest import ROOT
from armsparse_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(1, 8), (31, 64), (4096, 256), (5000, 2048), (100_000, 16)])
def test_sums_and_copy(m, n):
    x = torch.randint(-8, 9, (m, n), device="cuda", generator=torch.Generator("cuda").manual_seed(m)).float()
    y, s = kernels.to_bf16_colsum(x)
    assert s.dtype == torch.float32 and torch.equal(s, x.sum(0, dtype=torch.float64).float())
    assert torch.equal(y, x.to(torch.bfloat16))


def test_short_matrix_without_workspace():
    """Column sums of up to 4096 rows take no workspace by themselves: the pair does without, too."""
    code = ("import torch\nfrom armsparse_amd import kernels\nx = torch.ones(100, 64, device='cuda')\n"
            "y, s = kernels.to_bf16_colsum(x)\n"
            "assert bool((s == 100).all()) and torch.equal(y, x.to(torch.bfloat16))\nprint('held')\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=dict(os.environ, ARMSP_FAIL_ALLOC="1"),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "held" in r.stdout, r.stderr[-2000:]
