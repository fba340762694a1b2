"""The device radix sort behind csr_transpose and coo_to_csr at the sizes where it
changes: tile edges, the step from small to large tiles, one to three passes,
narrow digits.  Integer results, values moved or summed in input order: compared
bit for bit with numpy's stable sort."""
import numpy as np
import pytest
import torch

from armsparse_amd import kernels

pytestmark = pytest.mark.gpu

BIG = 2 << 20  # records from which tiles hold 16,384


def _csr(m, k, nnz, seed):
    """A CSR matrix with empty rows, hub rows and unsorted, repeated columns."""
    r = np.random.default_rng(seed)
    rows = np.sort((r.random(nnz) ** 3 * m).astype(np.int64))
    cols = (r.random(nnz) ** 2 * k).astype(np.int32)
    rp = np.zeros(m + 1, np.int32)
    np.cumsum(np.bincount(rows, minlength=m), out=rp[1:])
    return rp, cols, r.standard_normal(nnz).astype(np.float32), rows.astype(np.int32)


@pytest.mark.parametrize("values", [True, False])
@pytest.mark.parametrize("m,k,nnz", [
    (1, 1, 1), (3, 2, 2047), (70, 17, 2048), (5000, 1024, 2049), (9, 1025, 4097), (4000, (1 << 20) + 1, 30_000),
    (100_000, 3, 16_385), (50, 70_000, BIG - 1), (300_000, 300_007, BIG), (1 << 20, 1 << 20, BIG + 16_385),
    (70_000, 60_000, 20_000_000),  # more tiles than the scan holds counts of
])
def test_transpose_is_a_stable_sort(m, k, nnz, values):
    rp, ci, va, rows = _csr(m, k, nnz, m + k + nnz)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    cp, ri, vt = kernels.csr_transpose(dev(rp), dev(ci), dev(va) if values else None, k)
    order = np.argsort(ci, kind="stable")
    ref = np.zeros(k + 1, np.int64)
    np.cumsum(np.bincount(ci, minlength=k), out=ref[1:])
    assert np.array_equal(cp.cpu().numpy(), ref)
    assert np.array_equal(ri.cpu().numpy(), rows[order])
    assert vt is None if not values else np.array_equal(vt.cpu().numpy(), va[order])


@pytest.mark.parametrize("values,drop", [(True, False), (True, True), (False, True)])
@pytest.mark.parametrize("m,k,nnz", [(1, 1, 5), (2, 3000, 4095), (1025, 1023, 4097), (70_000, 5, 65_537),
                                     (2000, (1 << 20) + 3, 100_001), (300_007, 200_003, BIG + 1)])
def test_coo_to_csr_matches_numpy(m, k, nnz, values, drop):
    r = np.random.default_rng(nnz)
    rows, cols = r.integers(0, m, nnz).astype(np.int32), (r.random(nnz) ** 2 * k).astype(np.int32)
    va = r.integers(-2, 3, nnz).astype(np.float32)  # sums that cancel, exactly
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    rp, ci, vo = kernels.coo_to_csr(dev(rows), dev(cols), dev(va) if values else None, m, k, drop_zeros=drop)
    keys, inv = np.unique(rows.astype(np.int64) * k + cols, return_inverse=True)
    sums = np.bincount(inv, weights=va, minlength=keys.size).astype(np.float32)
    keep = sums != 0 if values and drop else np.ones(keys.size, bool)
    keys, sums = keys[keep], sums[keep]
    ref = np.zeros(m + 1, np.int64)
    np.cumsum(np.bincount(keys // k, minlength=m), out=ref[1:])
    assert np.array_equal(rp.cpu().numpy(), ref)
    assert np.array_equal(ci.cpu().numpy(), keys % k)
    assert vo is None if not values else np.array_equal(vo.cpu().numpy(), sums)


@pytest.mark.parametrize("bad", [(0, -1), (0, 50), (1, -5), (1, 40)])
def test_coo_out_of_range_index_writes_nothing(bad):
    r = np.random.default_rng(0)
    idx = [r.integers(0, 40, 5000).astype(np.int32), r.integers(0, 40, 5000).astype(np.int32)]
    idx[bad[0]][4321] = bad[1]
    from armsparse_amd import _lib
    rows, cols = (torch.from_numpy(a).cuda() for a in idx)
    out = [torch.full((n,), 7, dtype=torch.int32, device="cuda") for n in (41, 5000, 1)]
    with pytest.raises(_lib.ArmspError):
        _lib.call("armsp_coo_to_csr", 40, 40, 5000, kernels._ptr(rows), kernels._ptr(cols), None, 0,
                  kernels._ptr(out[0]), kernels._ptr(out[1]), None, kernels._ptr(out[2]), kernels._stream(rows.device))
    torch.cuda.synchronize()
    assert all(bool((t == 7).all()) for t in out)
