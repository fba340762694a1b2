"""Products written as bfloat16 and the conversions around them: the fp32 result rounded
once, bit for bit, at widths that take every kernel, with rows cut by chunk
boundaries, epilogues and unaligned operands."""
import numpy as np
import pytest
import torch

from armsparse_amd import _lib, kernels

pytestmark = pytest.mark.gpu


def graph(m, k, nnz, seed):
    r = np.random.default_rng(seed)
    rows = np.sort((r.random(nnz) ** 4 * m).astype(np.int64))  # hub rows of many chunks, empty rows
    rp = np.zeros(m + 1, np.int32)
    np.cumsum(np.bincount(rows, minlength=m), out=rp[1:])
    ci = r.integers(0, k, nnz).astype(np.int32)
    va = r.standard_normal(nnz).astype(np.float32)
    return [torch.from_numpy(a).cuda() for a in (rp, ci, va)]


@pytest.mark.parametrize("n", [3, 5, 8, 33, 64, 100, 128, 130, 192, 256, 320, 512])
@pytest.mark.parametrize("layout", ["packed", "pitched", "offset"])
def test_product_equals_the_rounded_fp32_product(n, layout):
    rp, ci, va = graph(900, 700, 30_000, n)
    b = torch.randn(700, n, device="cuda").to(torch.bfloat16)
    if layout == "pitched":
        buf = kernels.empty_rows(700, n, torch.bfloat16, "cuda")
        b = buf.copy_(b)
    elif layout == "offset":  # rows that start on no vector boundary
        b = torch.empty(700 * n + 1, dtype=torch.bfloat16, device="cuda")[1:].view(700, n).copy_(b)
    scale = torch.rand(900, device="cuda")
    for v in (va, None):
        for rs in (None, scale):
            want = kernels.spmm(rp, ci, v, b, row_scale=rs).to(torch.bfloat16)
            got = kernels.spmm_to_bf16(rp, ci, v, b, row_scale=rs)
            assert got.dtype == torch.bfloat16 and torch.equal(got, want)


def test_epilogue_and_refusals():
    rp, ci, va = graph(900, 700, 30_000, 1)
    b = torch.randn(700, 64, device="cuda").to(torch.bfloat16)
    bias, rs = torch.randn(64, device="cuda"), torch.rand(900, device="cuda")
    c = torch.empty(900, 64, dtype=torch.bfloat16, device="cuda")
    ep = _lib.Epilogue(None, rs.data_ptr(), bias.data_ptr(), 1)
    import ctypes
    p, s = kernels._ptr, kernels._stream(b.device)
    _lib.call("armsp_spmm_bf16_out", 900, 700, 64, ci.numel(), p(rp), p(ci), p(va), p(b), 64, p(c), 64,
              ctypes.byref(ep), s)
    want = kernels.spmm(rp, ci, va, b, row_scale=rs, bias=bias, relu=True).to(torch.bfloat16)
    assert torch.equal(c, want)
    for n, nnz in ((4, ci.numel()), (64, 0)):
        st = _lib.lib.armsp_spmm_bf16_out(900, 700, n, nnz, p(rp), p(ci), p(va), p(b), 64, p(c), 64, None, s)
        assert st == _lib.ERROR_NOT_SUPPORTED
    torch.cuda.synchronize()
    assert torch.equal(c, want)
    z = torch.zeros(901, dtype=torch.int32, device="cuda")
    assert not kernels.spmm_to_bf16(z, ci[:0], va[:0], b).any()


@pytest.mark.parametrize("m,n", [(1, 8), (31, 8), (33, 64), (4097, 256), (70_001, 128), (500, 2048), (300, 12), (5, 7)])
def test_conversions(m, n):
    x = torch.randn(m, n + 4, device="cuda")
    for t in (x[:, :n], x[:, :n].contiguous(), x[:, 1:n + 1]):
        want = t.to(torch.bfloat16)
        assert torch.equal(kernels.to_bf16(t, pitched=True), want)
        assert torch.equal(kernels.to_bf16(t, rows16=True), want)
        assert torch.equal(kernels.to_bf16(t), want)
    flat = x.reshape(-1)[1:]  # no 16-byte boundary
    assert torch.equal(kernels.to_bf16(flat), flat.to(torch.bfloat16))
    t = x[:, :n].contiguous()
    y, cs = kernels.to_bf16_colsum(t)
    assert torch.equal(y, t.to(torch.bfloat16))
    # fp32 sums of m terms in at most 64-term chains and two joins: a bound of 80 roundings of sum |x|
    err = (cs.double() - t.double().sum(0)).abs()
    assert bool((err <= 80 * 2.0 ** -24 * t.double().abs().sum(0)).all())
    assert torch.equal(kernels.to_bf16_colsum(t)[1], cs)
