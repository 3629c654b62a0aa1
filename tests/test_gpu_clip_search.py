"""GPU: the clip search's two-pass selection equals its exhaustive scan.

Rows whose scales lie outside [2^-24, 2^24] scan every candidate exactly.  With
norm 2 (and with Hessian-diagonal weights) the error of a row scaled by 2^-30
is the row's error scaled by 2^-60, so the search on the scaled rows, which
takes the exhaustive scan, must return the same zero points and the scales
times 2^-30, bit for bit.
"""
import pytest
import torch

from tests._util import gen

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("sym", [True, False])
@pytest.mark.parametrize("rows,cols,bits,grid,shrink", [
    (1, 1, 4, 50, 0.5), (3, 7, 2, 50, 0.5), (130, 32, 3, 50, 0.5), (5, 100, 8, 50, 0.5),
    (257, 128, 4, 50, 0.5), (6, 1000, 4, 32, 1.0), (9, 128, 4, 100, 0.8), (9, 64, 4, 10, 0.05)])
def test_selected_candidates_equal_exhaustive_scan(dev, rows, cols, bits, grid, shrink, sym,
                                                   weighted):
    from g2ptq_amd import WeightQuantizer
    print(f"clip search {rows}x{cols} W{bits} sym={sym} grid={grid} weighted={weighted}",
          flush=True)
    g = gen(77 + rows + cols)
    x = torch.randn(rows, cols, generator=g) * 0.02
    x[0, 0] = 0.3  # an outlier: the best clip is far from the range's end
    if rows > 4:
        x[1] = x[1].abs()                              # one-sided groups
        x[2] = -x[2].abs()
        x[3] = torch.round(x[3] * 200) / 64            # many equal errors
        x[4] = 0.0                                     # a zero scale
    x = x.to(dev)
    h = (torch.rand(1, cols, generator=g) + 0.1).to(dev) if weighted else None
    out = []
    for factor in (1.0, 2.0 ** -30):
        q = WeightQuantizer()
        q.configure(bits, perchannel=True, sym=sym, mse=True, norm=2.0, grid=grid,
                    maxshrink=shrink, hclip=weighted)
        flags = torch.zeros(1, dtype=torch.int32, device=dev)
        q.find_params(x * factor, h, _flags=flags)
        out.append((q.scale, q.zero, int(flags)))
    (s, z, f), (s30, z30, f30) = out
    assert torch.equal(s * 2.0 ** -30, s30)
    assert torch.equal(z.nan_to_num(nan=99.0), z30.nan_to_num(nan=99.0))
    assert f == f30
