"""Buffers that kernels fill with fp32 are fp32 whatever torch's default type is."""
import pytest
import torch

from armsparse_amd import kernels, op

pytestmark = pytest.mark.gpu


@pytest.fixture
def float64_default():
    torch.set_default_dtype(torch.float64)
    yield
    torch.set_default_dtype(torch.float32)


def test_sums_and_max_under_a_float64_default(float64_default):
    x = torch.arange(96, device="cuda", dtype=torch.float32).reshape(6, 16)
    for s in (kernels.colsum(x), kernels.to_bf16_colsum(x)[1]):
        assert s.dtype == torch.float32 and torch.equal(s, x.sum(0))
    rp = torch.tensor([0, 2, 2, 3], dtype=torch.int32, device="cuda")
    ci = torch.tensor([1, 5, 0], dtype=torch.int32, device="cuda")
    b = x.clone().requires_grad_(True)
    y = op.SPMMMaxFunction.apply(rp, ci, b)
    assert y.dtype == torch.float32 and torch.equal(y[0], x[5]) and torch.equal(y[2], x[0])
    y.sum().backward()
    assert b.grad.dtype == torch.float32 and b.grad[5].sum() == 16 and b.grad[0].sum() == 16 and b.grad.sum() == 32
