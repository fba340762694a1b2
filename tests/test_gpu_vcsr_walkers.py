"""Vector-aware CSR SpMV at the lengths where its walkers' loops turn: iterations of a
medium row, staging batches and reading steps of a long one, the limit between
them, and more rows than one listing workgroup holds.  Bit for bit with the
restated reference in both readings, signed zeros among the sums."""
import numpy as np
import pytest
import torch

import oracle
from armsparse_amd import data, kernels

pytestmark = pytest.mark.gpu


def blocked(nbs, K, seed):
    """Rows of exactly nbs[r] blocks, one nonzero each; every ninth value a signed zero."""
    r = np.random.default_rng(seed)
    cols = [4 * np.sort(r.choice(K // 4, n, replace=False)) + r.integers(0, 4, n) for n in nbs]
    rp = np.zeros(len(nbs) + 1, np.int32)
    rp[1:] = np.cumsum(nbs)
    va = r.uniform(-1, 1, rp[-1]).astype(np.float32)
    return data.csr_to_vcsr(data.CSR(rp, np.concatenate(cols).astype(np.int32), va, (len(nbs), K))), r


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("nbs", [
    [16, 17, 18, 19, 20, 31, 32, 33, 47, 48, 49, 64, 65],
    [17, 383, 0, 384, 385, 3, 386, 400, 17, 17, 300],
    [575, 576, 577, 192 * 3 + 15, 192 * 3 + 16, 192 * 3 + 17, 192 * 4 - 1, 192 * 4, 192 * 4 + 1, 3000, 3071, 3072, 3103, 3104, 4000],
    [1, 0, 2, 40, 0, 500] * 2000,
])
def test_walker_loops_are_bit_exact(nbs, fused):
    v, r = blocked(nbs, 1 << 14, len(nbs))
    assert list(np.diff(v.rowptr) // 4) == list(nbs)
    x = r.uniform(-1, 1, 1 << 14).astype(np.float32)
    x[r.random(x.size) < 0.1] = -0.0
    y0 = r.uniform(-1, 1, len(nbs)).astype(np.float32)
    y0[::3] = -0.0
    d = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (v.rowptr, v.colind, v.values, x, y0)]
    kernels.vcsr_spmv(*d, fused=fused)
    want = oracle.sparse_dense_vector(x, y0.copy(), v.rowptr, v.colind, v.values, fused=fused)
    assert np.array_equal(d[4].cpu().numpy().view(np.uint32), want.view(np.uint32))
