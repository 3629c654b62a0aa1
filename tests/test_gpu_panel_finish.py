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


def _shifted(t):
    """t's values one float off the 16-byte grid."""
    buf = torch.empty(t.numel() + 1, device=t.device, dtype=t.dtype)
    v = buf[1:].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize("B,C", [(1, 4), (2, 60), (1, 64), (3, 68), (2, 516), (1, 1600)])
def test_factor_copies_agree_off_the_vector_grid(dev, B, C):
    """The reversed copies of H and U on 16-byte steps and element by element:
    the same bits, damp included."""
    from g2ptq_amd import _core, _lib
    print(f"factor copies B={B} C={C}", flush=True)
    a = torch.randn(B, C, 2 * C, generator=gen(B + C), dtype=torch.float64)
    H = (a @ a.transpose(1, 2) / (2 * C)).float().to(dev)
    out = []
    for h in (H, _shifted(H)):
        U = torch.full_like(H, float("nan"))
        U = U if h is H else _shifted(U)
        info = torch.zeros(B, dtype=torch.int32, device=dev)
        ws = _lib.workspace(_lib.query_size("g2ptq_factor_workspace", B, C), dev)
        _lib.call("g2ptq_inv_chol_upper", _core.stream(), _lib.ptr(h), B, C, 0.0123, None,
                  _lib.ptr(U), _lib.ptr(info), _lib.ptr(ws), ws.numel())
        assert info.cpu().tolist() == [0] * B
        out.append(U.clone())
    assert torch.equal(out[0], out[1])
    assert torch.equal(out[0], out[0].triu()) and torch.isfinite(out[0]).all()


@pytest.mark.parametrize("C,gs", [(96, 32), (544, 32), (1032, 8)])
def test_transposed_factor_off_the_vector_grid(dev, C, gs):
    """Block tails from a factor transposed on 16-byte steps and element by
    element, values far from rounding ties: the same codes, and weights within
    128 fp32 roundings of the largest Σ|e·U| (below 0.12)."""
    from g2ptq_amd import _core, _lib
    print(f"transposed factor C={C}", flush=True)
    g, R, bs = gen(C), 37, 32
    W0 = (torch.randint(-6, 7, (1, R, C), generator=g) + 0.2 * torch.rand(1, R, C, generator=g)
          - 0.1) / 8
    W0[:, :, ::gs] = 7.5 / 8
    U = torch.triu(torch.randn(1, C, C, generator=g) * 1e-4, 1)
    U += torch.diag_embed(torch.rand(1, C, generator=g) * 0.5 + 0.75)
    out = []
    for shift in (False, True):
        W, Ud = W0.clone().to(dev), U.to(dev)
        Ud = _shifted(Ud) if shift else Ud
        Q, I, S = (torch.empty_like(W) for _ in range(3))
        st = torch.empty(-(-C // gs), R, device=dev)
        zt = torch.empty_like(st)
        flags = torch.zeros(1, dtype=torch.int32, device=dev)
        n = _lib.query_size("g2ptq_compensate_workspace", 0, 1, R, C, bs)
        ws = torch.empty(n, dtype=torch.uint8, device=dev)
        _lib.call("g2ptq_compensate", _core.stream(), 0, 1, R, C, bs, _lib.ptr(W), _lib.ptr(Ud),
                  None, None, None, 4, 1, gs, 0, 0, 0.0, 0.0, None, 0, None, _lib.ptr(st),
                  _lib.ptr(zt), _lib.ptr(Q), _lib.ptr(I), _lib.ptr(S), _lib.ptr(flags),
                  _lib.ptr(ws), n)
        torch.cuda.synchronize()
        out.append((W, I))
    assert torch.equal(out[0][1], out[1][1])
    assert (out[0][0] - out[1][0]).abs().max().item() <= 128 * 2.0 ** -24 * 0.12 + 4 * 2.0 ** -24
