"""Products of tensors of a subclass give plain tensors."""
import pytest
import torch

from armsparse_amd import kernels

pytestmark = pytest.mark.gpu


class Tagged(torch.Tensor):
    pass


def test_outputs_are_plain_tensors():
    rp = torch.tensor([0, 1, 3], dtype=torch.int32, device="cuda")
    ci = torch.tensor([1, 0, 1], dtype=torch.int32, device="cuda")
    va = torch.tensor([2.0, 1.0, 1.0], device="cuda")
    b = torch.arange(16.0, device="cuda").reshape(2, 8)
    for d in (b, b.as_subclass(Tagged), torch.nn.Parameter(b)):
        c = kernels.spmm(rp, ci, va, d)
        y = kernels.spmv(rp, ci, va, d[:, 3].detach().contiguous())
        assert type(c) is torch.Tensor and type(y) is torch.Tensor and not c.requires_grad
        assert torch.equal(c, torch.stack([2 * b[1], b[0] + b[1]])) and torch.equal(y, c[:, 3])
