"""Max aggregation at the sizes where its paths change: long rows cut over waves and joined
(more nonzeros than a workgroup per long row takes), a single row of them, the same without
workspace, and the backward pass with its table of lines.  Bit for bit with the fold."""
import numpy as np
import pytest
import torch

from armsparse_amd import kernels
from test_gpu_max import fold, matrix

pytestmark = pytest.mark.gpu


def dev(a):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()


# nonzeros times lanes per group on both sides of 2^19
@pytest.mark.parametrize("n,hub", [(1, 131_000), (1, 132_000), (3, 132_000), (8, 132_000), (33, 8000), (33, 9000), (64, 32_000),
                                   (64, 33_000), (66, 9000), (128, 17_000), (260, 9000)])
def test_cut_rows_with_special_values(n, hub):
    rp, ci, va = matrix([3, 0, 0, hub - 3000, 1, 0, 700, 64, 63, 65, 0, 128, 0] + [33, 1, 40, 0, 2] * 20, 97, n)
    r = np.random.default_rng(n)
    B = r.integers(-3, 4, (97, n)).astype(np.float32)
    special = np.array([np.nan, np.inf, -np.inf, -0.0, 0.0], np.float32)
    at = r.random(B.shape) < 0.02
    B[at] = special[r.integers(0, 5, int(at.sum()))]
    for v, init in ((None, kernels.MAX_INIT), (va, -np.inf)):
        out, arg = kernels.spmm_max(dev(rp), dev(ci), dev(v), dev(B), init=float(init), return_argmax=True)
        eo, ea = fold(rp, ci, v, B, init)
        out = out.cpu().numpy()
        assert np.array_equal(arg.cpu().numpy(), ea)
        nan = np.isnan(eo)
        assert np.array_equal(np.isnan(out), nan)
        assert np.array_equal(out[~nan].view(np.uint32), eo[~nan].view(np.uint32))


@pytest.mark.parametrize("n,length", [(64, 4099), (64, 40_000), (5, 9001)])
def test_the_only_row_among_empty_ones(n, length):
    rp, ci, va = matrix([0] * 50 + [length] + [0] * 100, 300, n)
    B = np.random.default_rng(n).standard_normal((300, n)).astype(np.float32)
    out, arg = kernels.spmm_max(dev(rp), dev(ci), dev(va), dev(B), return_argmax=True)
    eo, ea = fold(rp, ci, va, B, kernels.MAX_INIT)
    assert np.array_equal(out.cpu().numpy(), eo) and np.array_equal(arg.cpu().numpy(), ea)


@pytest.mark.parametrize("rows", [40, 4000])
def test_captured_without_an_arena(rows):
    """A captured call replays right, with workspace or without, on both sides of the limit."""
    rp, ci, _ = matrix([3, 0, 300, 2] * rows, 97, 1)
    d = [dev(a) for a in (rp, ci)]
    B = torch.randn(97, 96, device="cuda", generator=torch.Generator("cuda").manual_seed(rows))
    want, warg = kernels.spmm_max(*d, None, B, return_argmax=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out, arg = kernels.spmm_max(*d, None, B, return_argmax=True)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(arg, warg)


# outputs on both sides of 8192 per CU (256 CUs), from which workgroups collect adds in a table
@pytest.mark.parametrize("m,k,n", [(65_535, 3000, 32), (65_537, 3000, 32), (70_001, 5000, 33), (300, 700, 9001),
                                   (2_100_001, 50, 1), (40_000, 20, 64)])
def test_backward_with_a_table_of_lines(m, k, n):
    r = np.random.default_rng(m + n)
    nnz = 4 * m
    ci = (r.random(nnz) ** 4 * k).astype(np.int32)  # hub columns, and more lines than the table holds
    va = r.integers(-2, 3, nnz).astype(np.float32)  # integers: exact in any order
    g = r.integers(-3, 4, (m, n)).astype(np.float32)
    arg = r.integers(-1, nnz, (m, n)).astype(np.int32)
    for row, x in ((0, np.inf), (m // 2, np.nan), (m - 1, -np.inf)):  # each in a column of its own
        g[row, row % n] = x
    at = arg >= 0
    cols = np.broadcast_to(np.arange(n), (m, n))[at]
    for v in (None, va):
        with np.errstate(all="ignore"):
            add = g[at] if v is None else g[at] * v[arg[at]]
        key = ci[arg[at]].astype(np.int64) * n + cols
        odd = ~np.isfinite(add)
        want = np.bincount(key[~odd], weights=add[~odd], minlength=k * n).astype(np.float32)
        with np.errstate(all="ignore"):
            np.add.at(want, key[odd], add[odd])
        got = kernels.spmm_max_backward(dev(ci), dev(v), dev(g), dev(arg), k).cpu().numpy().reshape(-1)
        assert np.array_equal(got, want, equal_nan=True)
