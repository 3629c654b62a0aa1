"""GPU: the Cholesky panel's last step at edge sizes.

Panels of 512 columns, 64 at a time, over C just below, at and past one and two
panels, with rows that are not a multiple of 64 (nor of 4): U against torch's
fp64 inverse and Cholesky of a well-conditioned matrix.  Tolerance: a backward
stable fp32 factor of condition number kappa has a relative error of order
kappa·eps·C in the worst case; kappa is about 4 here.
"""
import pytest
import torch

from tests._util import gen

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


@pytest.mark.parametrize("C", [512, 513, 516, 575, 577, 1023, 1025, 1091, 1600])
def test_factor_at_panel_edges(dev, C):
    from tests.test_gpu_diag_block import _factor
    print(f"factor C={C}", flush=True)
    a = torch.randn(C, 4 * C, generator=gen(C), dtype=torch.float64)
    h = (a @ a.T / (4 * C)).float()
    ref = torch.linalg.cholesky(torch.linalg.inv(h.double()), upper=True)
    U, info = _factor(h.to(dev).unsqueeze(0), 0.0)
    assert info == [0]
    err = (U[0].double().cpu() - ref).norm() / ref.norm()
    assert err < 16 * 2.0 ** -24 * C ** 0.5, err
    assert torch.equal(U[0].cpu(), U[0].cpu().triu())
