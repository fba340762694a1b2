"""Sparse × sparse into dense at the edges of its tiles, windows and prefetch: bit for
bit with the restated reference."""
import numpy as np
import pytest
import torch

import oracle
from armsparse_amd import kernels

pytestmark = pytest.mark.gpu


def rows_of(lens, k, r):
    rp = np.zeros(len(lens) + 1, np.int32)
    rp[1:] = np.cumsum(lens)
    ci = [np.sort(r.choice(k, n, replace=False)) for n in lens]
    return rp, np.concatenate(ci).astype(np.int32), r.uniform(-1, 1, rp[-1]).astype(np.float32)


@pytest.mark.parametrize("n", [1, 64, 2047, 2048, 2049, 4100, 6147])
@pytest.mark.parametrize("offset", [0, 1])
def test_tile_and_window_edges(n, offset):
    r = np.random.default_rng(n)
    k = 200
    a = rows_of([0, 1, 2, 7, 8, 9, 15, 16, 17, 63, 64, 65, 72, 128, 129, 200, 0], k, r)
    b = rows_of(np.minimum(r.choice([0, 1, 3, 20, 63, 64, 65, 130], k), n), n, r)
    c0 = r.uniform(-1, 1, (17, n)).astype(np.float32)
    d = lambda t: tuple(torch.from_numpy(x).cuda() for x in t)  # noqa: E731
    c = torch.empty(17 * n + 1, device="cuda")[offset:offset + 17 * n].view(17, n)  # offset 1: no 16-byte rows
    c.copy_(torch.from_numpy(c0))
    kernels.spgemm_dense(d(a), d(b), c)
    want = oracle.sparse_matrix_mul3(a, b, c0.copy())
    assert np.array_equal(c.cpu().numpy().view(np.uint32), want.view(np.uint32))
