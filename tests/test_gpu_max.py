"""Max aggregation over cut rows: hub rows many chunks long, rows that end on chunk
boundaries, empty rows, NaN, infinities and signed zeros, every column width of the
kernels, with and without workspace.  The fold's results bit for bit."""
import numpy as np
import pytest
import torch

from armsparse_amd import kernels

pytestmark = pytest.mark.gpu


def fold(rp, ci, va, B, init):
    out = np.full((len(rp) - 1, B.shape[1]), np.float32(init), np.float32)
    arg = np.full(out.shape, -1, np.int32)
    with np.errstate(all="ignore"):
        for r in range(len(rp) - 1):
            for p in range(rp[r], rp[r + 1]):
                x = B[ci[p]] if va is None else np.float32(va[p]) * B[ci[p]]
                take = ~(out[r] > x)
                out[r] = np.where(take, x, out[r])
                arg[r] = np.where(take, p, arg[r])
    return out, arg


def matrix(lens, k, seed):
    rp = np.zeros(len(lens) + 1, np.int32)
    np.cumsum(lens, out=rp[1:])
    r = np.random.default_rng(seed)
    return rp, r.integers(0, k, rp[-1]).astype(np.int32), r.standard_normal(rp[-1]).astype(np.float32)


SHAPES = {
    "hub": [3, 0, 0, 5000, 1, 0, 700, 64, 63, 65, 0],
    "one row": [4099],
    "boundaries": [63, 63, 127, 0, 63] * 20,
    "short": [0, 1, 2, 0, 0, 3, 7, 8, 9] * 40,
}


@pytest.mark.parametrize("n", [1, 3, 33, 64, 65, 66, 128, 132, 256, 260])
@pytest.mark.parametrize("shape", SHAPES)
def test_cut_rows_with_special_values(shape, n):
    rp, ci, va = matrix(SHAPES[shape], 97, n)
    r = np.random.default_rng(n)
    B = r.integers(-3, 4, (97, n)).astype(np.float32)  # ties: the later position must win
    special = np.array([np.nan, np.inf, -np.inf, -0.0, 0.0], np.float32)
    at = r.random(B.shape) < 0.02
    B[at] = special[r.integers(0, 5, int(at.sum()))]
    d = lambda a: None if a is None else torch.from_numpy(a).cuda()  # noqa: E731
    for v, init in ((None, kernels.MAX_INIT), (va, -np.inf), (va, 1.5)):
        out, arg = kernels.spmm_max(d(rp), d(ci), d(v), d(B), init=float(init), return_argmax=True)
        eo, ea = fold(rp, ci, v, B, init)
        out = out.cpu().numpy()
        assert np.array_equal(arg.cpu().numpy(), ea)
        nan = np.isnan(eo)
        assert np.array_equal(np.isnan(out), nan)
        assert np.array_equal(out[~nan].view(np.uint32), eo[~nan].view(np.uint32))
        only = kernels.spmm_max(d(rp), d(ci), d(v), d(B), init=float(init)).cpu().numpy()
        assert np.array_equal(only.view(np.uint32), out.view(np.uint32))


def test_capture_without_an_arena_runs_without_workspace():
    """A captured call that finds no workspace still runs (a group of lanes per row)."""
    rp, ci, _ = matrix([3, 0, 900, 2] * 600, 97, 1)
    d = [torch.from_numpy(a).cuda() for a in (rp, ci)]
    B = torch.randn(97, 640, device="cuda")
    want, warg = kernels.spmm_max(*d, None, B, return_argmax=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out, arg = kernels.spmm_max(*d, None, B, return_argmax=True)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(arg, warg)


@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (31, 9, 31), (33, 70, 32), (70, 33, 33), (1000, 97, 130), (257, 300, 300)])
def test_backward_adds_into_the_winning_rows(m, k, n):
    r = np.random.default_rng(m + n)
    nnz = 5 * m
    ci = r.integers(0, k, nnz).astype(np.int32)
    va = r.integers(-2, 3, nnz).astype(np.float32)  # integers: exact in any order
    g = r.integers(-3, 4, (m, n)).astype(np.float32)
    arg = r.integers(-1, nnz, (m, n)).astype(np.int32)
    d = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    for v in (None, va):
        want = np.zeros((k, n), np.float32)
        rows, cols = np.nonzero(arg >= 0)
        p = arg[rows, cols]
        np.add.at(want, (ci[p], cols), g[rows, cols] * (1 if v is None else v[p]))
        got = kernels.spmm_max_backward(d(ci), None if v is None else d(v), d(g), d(arg), k)
        assert np.array_equal(got.cpu().numpy(), want)
