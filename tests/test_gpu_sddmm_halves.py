"""SDDMM at widths that are not whole steps of the kernel (32 fp32 or 64 bf16 columns), or
whole steps that have no middle: which of them an automatic call splits into column halves,
the values, and that the columns past the width leave no trace."""
import numpy as np
import pytest
import torch

from armsparse_amd import data, kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kd,dtype,split", [(160, torch.float32, False), (224, torch.float32, False),
                                            (320, torch.bfloat16, False), (176, torch.float32, True),
                                            (192, torch.float32, True), (352, torch.bfloat16, True)])
def test_automatic_choice_on_skewed_columns(kd, dtype, split):
    a = data.rmat_csr(18, 1 << 23, seed=9)
    rp, ci = (torch.from_numpy(x).cuda() for x in (a.rowptr, a.colind))
    gen = torch.Generator("cuda").manual_seed(kd)
    U, V = (torch.randn(1 << 18, kd, device="cuda", generator=gen).to(dtype) for _ in range(2))
    auto = kernels.sddmm(rp, ci, U, V)
    whole, halves = (kernels.sddmm(rp, ci, U, V, config=dict(schedule="merge", unroll=u)) for u in (1, 2))
    assert torch.equal(auto, halves if split else whole) and not torch.equal(whole, halves)
    at = torch.randint(1 << 23, (20_000,), device="cuda", generator=gen)
    rows = torch.searchsorted(rp, at.int(), right=True) - 1
    u, v = U[rows].double(), V[ci[at].long()].double()
    want, bound = (u * v).sum(1), (u * v).abs().sum(1)
    for out in (whole, halves):  # fp32 sums of kd products
        assert bool(((out[at].double() - want).abs() <= kd * 2.0 ** -24 * bound).all())


@pytest.mark.parametrize("unroll", [1, 2])
@pytest.mark.parametrize("kd,dtype", [(36, torch.float32), (136, torch.float32), (72, torch.bfloat16),
                                      (272, torch.bfloat16)])
def test_infinite_first_column(kd, dtype, unroll):
    """Lanes past the width load the first column; its infinities must not reach the sum."""
    a = data.uniform_csr(300, 200, 3000, seed=kd)
    rp, ci = (torch.from_numpy(x).cuda() for x in (a.rowptr, a.colind))
    U, V = torch.ones(300, kd, device="cuda").to(dtype), torch.ones(200, kd, device="cuda").to(dtype)
    V[:, 0] = float("inf")
    V[:, kd // 2:kd // 2 + 1] = 0.0
    out = kernels.sddmm(rp, ci, U, V, config=dict(schedule="merge", unroll=unroll)).cpu().numpy()
    assert np.all(np.isposinf(out))
