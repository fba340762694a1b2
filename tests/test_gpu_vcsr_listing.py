"""The listing of medium and long VCSR rows by workgroups of 1, 2, 4 and 8 rows a thread:
tall matrices with a few such rows at the edges of workgroups, bit for bit."""
import numpy as np
import pytest
import torch

from armsparse_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1 << 18, (1 << 18) + 1, (1 << 19) + 5, (1 << 22) + 9])
def test_few_long_rows_in_tall_matrices(m):
    r = np.random.default_rng(m)
    blocks = np.zeros(m, np.int64)
    blocks[r.integers(0, m, 1000)] = r.integers(0, 40, 1000)
    for at, n in ((0, 17), (1023, 70), (1024, 300), (2047, 129), (2048, 2100), (4095, 65), (8191, 16), (8192, 257), (m - 1, 4000)):
        blocks[at] = n
    rp = np.zeros(m + 1, np.int64)
    np.cumsum(4 * blocks, out=rp[1:])
    nb = int(rp[-1]) // 4
    ci = (4 * r.integers(0, 500, nb)[:, None] + np.arange(4)).reshape(-1).astype(np.int32)
    va, x = (r.standard_normal(k).astype(np.float32) for k in (4 * nb, 2000))
    y = r.standard_normal(m).astype(np.float32)
    want = y.copy()
    prod = (va * x[ci]).reshape(-1, 4)
    for row in np.nonzero(blocks)[0]:
        s = np.zeros(4, np.float32)
        for t in prod[rp[row] // 4:rp[row + 1] // 4]:
            s = s + t
        want[row] += (s[0] + s[2]) + (s[1] + s[3])
    d = [torch.from_numpy(a).cuda() for a in (rp.astype(np.int32), ci, va, x, y)]
    got = kernels.vcsr_spmv(*d).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
