"""GPU: the factor's 64x64 diagonal blocks at panel edges and ragged widths.

A matrix whose reversed pivot r is negative reports r + 1 (g2ptq_hip.h: the
leading minor that is not positive definite), whichever 16-column panel of a
diagonal block the pivot falls in; a tridiagonal matrix's factor is held to
fp64 within the first-order bound of its C sequential updates.
"""
import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


def _factor(H, percdamp):
    from g2ptq_amd import _core, _lib
    B, C, _ = H.shape
    U = torch.empty_like(H)
    info = torch.zeros(B, dtype=torch.int32, device=H.device)
    ws = _lib.workspace(_lib.query_size("g2ptq_factor_workspace", B, C), H.device)
    _lib.call("g2ptq_inv_chol_upper", _core.stream(), _lib.ptr(H), B, C, percdamp, None,
              _lib.ptr(U), _lib.ptr(info), _lib.ptr(ws), ws.numel())
    return U, info.cpu().tolist()


@pytest.mark.parametrize("C", [1, 15, 16, 17, 64, 65, 100, 200])
def test_failing_pivot_is_reported(dev, C):
    print(f"failing pivots C={C}", flush=True)
    bad = sorted({r for r in (0, 1, 15, 16, 31, 32, 47, 48, 63, 64, 79, 99, 150, C - 1) if r < C})
    H = torch.eye(C, device=dev).repeat(len(bad) + 1, 1, 1)
    for b, r in enumerate(bad):
        H[b, C - 1 - r, C - 1 - r] = -2.0
    U, info = _factor(H, 1e-6 if C > 3 else 0.0)
    assert info[:-1] == [r + 1 for r in bad]
    assert info[-1] == 0 and torch.isfinite(U[-1]).all()


@pytest.mark.parametrize("C", [1, 16, 17, 33, 63, 64, 65, 130])
def test_factor_of_a_tridiagonal_matrix(dev, C):
    print(f"tridiagonal factor C={C}", flush=True)
    d = torch.linspace(2.0, 3.0, C, dtype=torch.float64)
    A = torch.diag(d) + torch.diag(torch.full((C - 1,), -0.9, dtype=torch.float64), 1) \
        + torch.diag(torch.full((C - 1,), -0.9, dtype=torch.float64), -1)
    U, info = _factor(A.float().unsqueeze(0).to(dev), 0.0)
    assert info == [0]
    Ue = torch.linalg.cholesky(torch.linalg.inv(A.float().double()), upper=True)
    # cond(A) < 4: each entry carries at most a few roundings per earlier pivot
    err = (U[0].double().cpu() - Ue).abs().max().item()
    assert err <= 4 * (C + 4) * 2.0 ** -24, err
