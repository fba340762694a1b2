"""Sparse × sparse into dense with long B rows on both sides of the widths that take tiles of
4096 columns: bit for bit with the restated reference."""
import numpy as np
import pytest
import torch

import oracle
from armsparse_amd import kernels
from test_gpu_spgemm_tiles import rows_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16_384, 16_385, 20_480, 24_577, 65_536, 65_537])
@pytest.mark.parametrize("each", [299, 301, 420])
def test_wide_products(n, each):
    r = np.random.default_rng(n + each)
    k = 40
    a = rows_of([0, 1, 7, 8, 9, 40, 0, 17], k, r)
    b = rows_of([each] * (k - 2) + [each - 64, each + 64], n, r)
    c0 = r.uniform(-1, 1, (8, n)).astype(np.float32)
    d = lambda t: tuple(torch.from_numpy(x).cuda() for x in t)  # noqa: E731
    c = torch.from_numpy(c0).cuda()
    kernels.spgemm_dense(d(a), d(b), c)
    want = oracle.sparse_matrix_mul3(a, b, c0.copy())
    assert np.array_equal(c.cpu().numpy().view(np.uint32), want.view(np.uint32))
