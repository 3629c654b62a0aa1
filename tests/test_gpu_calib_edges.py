"""GPU: the calibration statistics on 16-byte steps and off them.

Group sizes that are and are not multiples of 8, offset pointers and short rows;
saliencies against fp64 (a sum of n squares in any order is within (n/8 + 16)
roundings), the running mean bit for bit against its expression evaluated by
torch.
"""
import numpy as np
import pytest
import torch

from tests._util import gen

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]
DTYPES = [torch.bfloat16, torch.float16, torch.float32]


@pytest.mark.parametrize("dtype", DTYPES, ids=["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("rows,groups,gs,offset", [(1, 1, 8, 0), (3, 2, 8, 0), (5, 4, 1024, 0),
                                                   (7, 1, 520, 0), (2, 3, 7, 0), (9, 2, 1000, 1),
                                                   (130, 4, 504, 0)])
def test_group_mean_square(dev, dtype, rows, groups, gs, offset):
    from g2ptq_amd.calib_utils import group_mean_square
    print(f"group mean square {rows}x{groups}x{gs}+{offset} {dtype}", flush=True)
    x = torch.randn(rows * groups * gs + offset, generator=gen(gs + rows)).to(dtype).to(dev)
    x = x[offset:].view(rows, groups * gs)
    out = group_mean_square(x, groups).double().cpu()
    exact = x.double().cpu().pow(2).view(rows, groups, gs).mean(-1)
    assert ((out - exact).abs() / exact).max().item() <= (gs / 8 + 16) * 2.0 ** -24


@pytest.mark.parametrize("dtype", DTYPES, ids=["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("gs", [8, 16, 32, 64, 120])
def test_narrow_groups_take_one_value_per_lane(dev, dtype, gs):
    """Groups under 128 values, where eight per lane are slower: the same sums in
    the same order as off the 16-byte grid, bit for bit."""
    from g2ptq_amd.calib_utils import group_mean_square
    print(f"narrow groups of {gs} {dtype}", flush=True)
    x = torch.randn(33 * 4 * gs, generator=gen(gs)).to(dtype).to(dev)
    off = torch.empty(x.numel() + 1, dtype=dtype, device=dev)[1:]
    off.copy_(x)
    assert torch.equal(group_mean_square(x.view(33, 4 * gs), 4),
                       group_mean_square(off.view(33, 4 * gs), 4))


@pytest.mark.parametrize("dtype", DTYPES, ids=["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("n,offset", [(8, 0), (24, 0), (7, 0), (4096, 0), (4097, 0), (4096, 1)])
def test_running_mean(dev, dtype, n, offset):
    from g2ptq_amd.calib_utils import running_mean_update
    print(f"running mean n={n}+{offset} {dtype}", flush=True)
    g = gen(n)
    cache = want = None
    for k in range(3):
        grad = torch.randn(n + offset, generator=g).to(dtype).to(dev)[offset:]
        cache = running_mean_update(cache, grad, 37, k)
        d = grad.float() * float(np.float32(1.0) / np.float32(37 * (k + 1)))
        want = d if want is None else want * float(np.float32(k / (k + 1))) + d
        assert torch.equal(cache, want), k
