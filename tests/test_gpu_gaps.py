"""Matrices with long runs of empty rows: the results, and that a run in the middle of the
matrix costs a call no more than one at its end."""
import numpy as np
import pytest
import torch

from armsparse_amd import kernels

pytestmark = pytest.mark.gpu


def gap(m, rows_each, k, seed, middle):
    """A matrix of m rows: rows_each of 0 to 59 entries at the start, as many after a run of
    empty rows that lies between the two (middle) or after both."""
    r = np.random.default_rng(seed)
    lens = np.zeros(m, np.int64)
    lens[:rows_each] = r.integers(0, 60, rows_each)
    second = slice(m - rows_each, m) if middle else slice(rows_each, 2 * rows_each)
    lens[second] = r.integers(0, 60, rows_each)
    rp = np.zeros(m + 1, np.int32)
    np.cumsum(lens, out=rp[1:])
    return rp, r.integers(0, k, rp[-1]).astype(np.int32), r.standard_normal(rp[-1]).astype(np.float32)


def best_ms(fn, n=5):
    t = []
    for _ in range(n):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        fn()
        b.record()
        b.synchronize()
        t.append(a.elapsed_time(b))
    return min(t)


def dev(*arrays):
    return [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in arrays]


def test_max_over_a_run_of_empty_rows():
    m, each, k, n = 4_000_000, 1000, 300, 4
    times = []
    for middle in (False, True):
        rp, ci, va = gap(m, each, k, 5, middle)
        B = np.random.default_rng(1).standard_normal((k, n)).astype(np.float32)
        d = dev(rp, ci, va, B)
        out, arg = kernels.spmm_max(*d, return_argmax=True)
        want, warg = np.full((m, n), np.float32(kernels.MAX_INIT)), np.full((m, n), -1, np.int32)
        for r in np.nonzero(np.diff(rp))[0]:
            x = va[rp[r]:rp[r + 1], None] * B[ci[rp[r]:rp[r + 1]]]
            at = len(x) - 1 - np.argmax(x[::-1], 0)  # the last of the largest
            want[r], warg[r] = x[at, np.arange(n)], rp[r] + at
        assert np.array_equal(out.cpu().numpy(), want) and np.array_equal(arg.cpu().numpy(), warg)
        times.append(best_ms(lambda: kernels.spmm_max(*d)))
    print("run of empty rows at the end, in the middle: %.3f, %.3f ms" % tuple(times))
    assert times[1] <= 3 * times[0]


def transposed(rp, ci, va, k):
    order = np.argsort(ci, kind="stable")
    cp = np.zeros(k + 1, np.int32)
    np.cumsum(np.bincount(ci, minlength=k), out=cp[1:])
    rows = np.repeat(np.arange(len(rp) - 1, dtype=np.int32), np.diff(rp))
    return cp, rows[order], va[order]


def test_transpose_over_a_run_of_empty_rows():
    m, each, k = 4_000_000, 1000, 300
    times = []
    for middle in (False, True):
        rp, ci, va = gap(m, each, k, 5, middle)
        d = dev(rp, ci, va)
        for got, want in zip(kernels.csr_transpose(*d, k), transposed(rp, ci, va, k)):
            assert np.array_equal(got.cpu().numpy(), want)
        times.append(best_ms(lambda: kernels.csr_transpose(*d, k)))
    print("run of empty rows at the end, in the middle: %.3f, %.3f ms" % tuple(times))
    assert times[1] <= 3 * times[0]


@pytest.mark.parametrize("nnz,rows_per_entry", [(n, q) for n in (1, 2047, 2049, 70_000) for q in (7, 8, 9, 100)] +
                         [((2 << 20) + n, q) for n in (5, 4095) for q in (23, 25)])
def test_transpose_of_mostly_empty_rows(nnz, rows_per_entry):
    """Tiles on both sides of the number of rows from which records search for theirs."""
    m, k = nnz * rows_per_entry, 1500
    r = np.random.default_rng(nnz)
    rp = np.zeros(m + 1, np.int32)
    np.cumsum(np.bincount(r.integers(0, m, nnz), minlength=m), out=rp[1:])
    ci, va = r.integers(0, k, nnz).astype(np.int32), r.standard_normal(nnz).astype(np.float32)
    for got, want in zip(kernels.csr_transpose(*dev(rp, ci, va), k), transposed(rp, ci, va, k)):
        assert np.array_equal(got.cpu().numpy(), want)
