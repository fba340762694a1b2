"""Merge-path kernels around the number of chunks from which a partition is computed, the
chunks that an automatic SpMM takes, and the column split of an automatic SDDMM."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from armsparse_amd import _lib, data, kernels

pytestmark = pytest.mark.gpu
TOL = 1e-5  # of the sum of absolute products, as in the other tests of these kernels


def dev(*arrays):
    return [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in arrays]


@pytest.mark.parametrize("waves", [4095, 4096, 4097])
@pytest.mark.parametrize("n", [1, 3, 20, 100])
def test_partition_threshold(waves, n):
    chunk = 256
    m = 30_000
    a = data.uniform_csr(m, 5000, waves * chunk - m - 7, seed=waves)
    r = np.random.default_rng(n)
    B = r.uniform(-1, 1, (5000, n)).astype(np.float32)
    U = r.uniform(-1, 1, (m, 32)).astype(np.float32)
    V = r.uniform(-1, 1, (5000, 32)).astype(np.float32)
    rp, ci, va, d_B, d_U, d_V = dev(a.rowptr, a.colind, a.values, B, U, V)
    ref = oracle.spmm_f64(a.rowptr, a.colind, a.values, B)
    bound = oracle.spmm_f64(a.rowptr, a.colind, np.abs(a.values), np.abs(B))
    cfg = dict(schedule="merge", chunk=chunk)
    out = kernels.spmm(rp, ci, va, d_B, config=cfg).cpu().numpy()
    assert np.all(np.abs(out - ref) <= TOL * bound + 1e-30)
    if n == 1:
        y = kernels.spmv(rp, ci, va, d_B[:, 0].contiguous(), config=cfg).cpu().numpy()
        assert np.all(np.abs(y - ref[:, 0]) <= TOL * bound[:, 0] + 1e-30)
        d = kernels.sddmm(rp, ci, d_U, d_V, config=cfg).cpu().numpy()
        dref = oracle.sddmm_f64(a.rowptr, a.colind, U, V)
        dbound = oracle.sddmm_f64(a.rowptr, a.colind, np.abs(U), np.abs(V))
        assert np.all(np.abs(d - dref) <= TOL * dbound + 1e-30)


@pytest.mark.parametrize("n", [8, 65, 100, 192])
def test_automatic_chunks(n):
    a = data.rmat_csr(17, 2_100_000, seed=n)
    B = np.random.default_rng(n).uniform(-1, 1, (a.shape[1], n)).astype(np.float32)
    rp, ci, va, d_B = dev(a.rowptr, a.colind, a.values, B)
    out = kernels.spmm(rp, ci, va, d_B).cpu().numpy()
    ref = oracle.spmm_f64(a.rowptr, a.colind, a.values, B)
    bound = oracle.spmm_f64(a.rowptr, a.colind, np.abs(a.values), np.abs(B))
    assert np.all(np.abs(out - ref) <= TOL * bound + 1e-30)


def test_allocation_free_product_takes_longer_chunks_where_short_ones_do_not_fit():
    """2.2M items, N = 3000: the carries of 512-item chunks fit the array, those of 256 do not."""
    a = data.uniform_csr(100_000, 1000, 2_100_000, seed=3)
    rp, ci, va = dev(a.rowptr, a.colind, a.values)
    B = torch.randn(1000, 3000, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    outs = []
    for fn in ("armsp_spmm_f32", "armsp_spmm_f32_noalloc"):
        C = torch.empty(100_000, 3000, device="cuda")
        assert getattr(_lib.lib, fn)(100_000, 1000, 3000, ci.numel(), p(rp), p(ci), p(va), p(B), 3000, p(C), 3000, 0,
                                     None, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        outs.append(C)
    assert torch.equal(outs[0].view(torch.int32), outs[1].view(torch.int32))


@pytest.mark.parametrize("kd,dtype,pad", [(128, torch.float32, 0), (136, torch.float32, 4), (256, torch.bfloat16, 0),
                                          (272, torch.bfloat16, 8)])
@pytest.mark.parametrize("kind", ["rmat", "uniform"])
def test_automatic_sddmm_split(kind, kd, dtype, pad):
    """On skewed columns the automatic call is the split one, on uniform ones the unsplit
    one, bit for bit; with and without a scale."""
    a = (data.rmat_csr(18, 1 << 23, seed=9) if kind == "rmat" else data.uniform_csr(1 << 18, 1 << 18, 1 << 23, seed=9))
    rp, ci, va = dev(a.rowptr, a.colind, a.values)
    gen = torch.Generator("cuda").manual_seed(kd)
    U, V = (torch.randn(1 << 18, kd + pad, device="cuda", generator=gen).to(dtype)[:, :kd] for _ in range(2))
    split = dict(schedule="merge", unroll=2 if kind == "rmat" else 1)
    for scale in (va, None):
        auto = kernels.sddmm(rp, ci, U, V, scale=scale)
        assert torch.equal(auto, kernels.sddmm(rp, ci, U, V, scale=scale, config=split))
    other = kernels.sddmm(rp, ci, U, V, config=dict(schedule="merge", unroll=1 if kind == "rmat" else 2))
    assert not torch.equal(auto, other)
