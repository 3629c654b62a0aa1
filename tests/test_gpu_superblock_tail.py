"""GPU: GPTQ's super-block launch (near tails on fp32 MFMAs in the sweep) at row
and column remainders.

The launch's blocks receive Σ_k e_k·U[k, c] as two ascending chains of fused
multiply-adds (even and odd k) added together; a run with one-block super-blocks
(a workspace for one block's errors) applies the same sums as split products.
Weights far from rounding ties therefore get the same codes, and the values that
both write agree within the products' bound: 128 fp32 roundings of Σ|e·U|.
"""
import pytest
import torch

from tests._util import gen

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


@pytest.mark.parametrize("B,R,C,sym", [(1, 1, 512, 1), (1, 15, 1024, 0), (1, 17, 384, 1),
                                       (2, 16, 640, 1), (3, 37, 1152, 0), (1, 200, 512, 1)])
def test_superblock_tail_matches_block_tails(dev, B, R, C, sym):
    from g2ptq_amd import _core, _lib
    print(f"super-block tail B={B} R={R} C={C}", flush=True)
    g = gen(B * 1000 + R + C)
    maxq, bs, gs = 7, 128, 128
    # group scales near 1/8 (sym: largest value 7.5/8, whose code is 7 on either
    # side of its tie; asym: range [-7/8, 8/8], zero point -1, no tie) and values
    # near the middle of their steps with small couplings: no code is at a tie
    W0 = (torch.randint(-6, 7, (B, R, C), generator=g) + 0.2 * torch.rand(B, R, C, generator=g) - 0.1) / 8
    W0[:, :, ::gs] = 7.5 / 8 if sym else 1.0
    if not sym:
        W0[:, :, 1::gs] = -7 / 8
    U = torch.triu(torch.randn(B, C, C, generator=g) * 1e-4, 1)
    U += torch.diag_embed(torch.rand(B, C, generator=g) * 0.5 + 0.75)
    out = []
    for full in (True, False):
        W, Ud = W0.clone().to(dev), U.to(dev)
        Q, I, S = (torch.empty_like(W) for _ in range(3))
        st = torch.empty(-(-C // gs), B * R, device=dev)
        zt = torch.empty_like(st)
        flags = torch.zeros(1, dtype=torch.int32, device=dev)
        n = _lib.query_size("g2ptq_compensate_workspace", 0, B, R, C, bs) if full else \
            (B * R * bs * 4 + 255) // 256 * 256
        ws = torch.empty(n, dtype=torch.uint8, device=dev)
        _lib.call("g2ptq_compensate", _core.stream(), 0, B, R, C, bs, _lib.ptr(W), _lib.ptr(Ud),
                  None, None, None, 4, sym, gs, 0, 0, 0.0, 0.0, None, 0, None, _lib.ptr(st),
                  _lib.ptr(zt), _lib.ptr(Q), _lib.ptr(I), _lib.ptr(S), _lib.ptr(flags),
                  _lib.ptr(ws), n)
        torch.cuda.synchronize()
        out.append((W, Q, I, st))
    (Wa, Qa, Ia, sa), (Wb, Qb, Ib, sb) = out
    assert torch.equal(Ia, Ib)
    # |e| <= 0.1, |U| <= 1e-3: Σ|e·U| over 512 columns is below 0.06
    tol = 128 * 2.0 ** -24 * 0.06 + 4 * 2.0 ** -24
    assert (Wa - Wb).abs().max().item() <= tol
    assert (sa - sb).abs().max().item() <= tol
    assert torch.allclose(Qa, Qb, rtol=0, atol=16 * tol)
