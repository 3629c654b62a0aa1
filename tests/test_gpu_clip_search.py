"""GPU: the clip search's two-pass selection equals its exhaustive scan.

Rows whose scales lie outside [2^-24, 2^24] scan every candidate exactly.  With
norm 2 (and with Hessian-diagonal weights) the error of a row scaled by 2^-30
is the row's error scaled by 2^-60, so the search on the scaled rows, which
takes the exhaustive scan, must return the same zero points and the scales
times 2^-30, bit for bit.  At other norms the parameters found are held to the
least error over all candidates, evaluated in fp64.
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


@pytest.mark.parametrize("cols,steps,sym,weighted", [
    (128, 1, True, False), (128, 1, False, True), (512, 1, False, False), (16, 1, True, False),
    (128, 2, False, False), (512, 2, True, False), (128, 3, True, True), (512, 3, False, True)])
def test_few_candidates_take_no_longer_than_the_scan(dev, cols, steps, sym, weighted):
    """A search of a few candidates is not bracketed first: it takes what the
    rows above the bounds' range take, which are scanned (bracketing made it 1.2
    to 5 times)."""
    from g2ptq_amd import _core, _lib
    rows = (1 << 23) // max(cols, 64)
    g = gen(cols + steps)
    x = (torch.randn(rows, cols, generator=g) * 0.02).to(dev)
    h = (torch.rand(1, cols, generator=g) + 0.1).to(dev) if weighted else None
    s, z = torch.empty(rows, device=dev), torch.empty(rows, device=dev)
    flags = torch.zeros(1, dtype=torch.int32, device=dev)

    def us(v, n=20):
        best = float("inf")
        for _ in range(4):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(n):
                _lib.call("g2ptq_find_params_mse", _core.stream(), _lib.ptr(v), rows, cols, cols, 4,
                          int(sym), 2.0, 10, (steps + 0.5) / 10, _lib.ptr(h), cols,
                          1 if weighted else 0, 1, _lib.ptr(s), _lib.ptr(z), 1, _lib.ptr(flags))
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) / n * 1e3)
        return best
    huge = x * 2.0 ** 42
    assert huge.abs().amax(1).min() >= 2.0 ** 34  # no row can be bracketed
    search, scan = us(x), us(huge)
    print(f"{steps}x{steps} candidates, groups of {cols}, sym={sym} weighted={weighted}: "
          f"{search:.1f} us, the scan {scan:.1f} us", flush=True)
    assert search <= 1.15 * scan


def _candidates(x, bits, sym, grid, steps):
    """Scale and zero (rows, 1) of every candidate, formed in fp32 as the search
    forms them (divisors as tensors: torch multiplies by a number's reciprocal)."""
    half = 2 ** (bits - 1)
    xmin, xmax = x.amin(1, keepdim=True).clamp_max(0), x.amax(1, keepdim=True).clamp_min(0)
    for i in range(steps):
        for j in range(steps):
            lo, hi = (1 - i / grid) * xmin, (1 - j / grid) * xmax
            if sym:
                s = torch.maximum(lo.abs(), hi) / torch.full_like(lo, (2 * half - 1) / 2)
                yield s, torch.zeros_like(s)
            else:
                s = (hi - lo) / torch.full_like(lo, 2 * half - 1)
                yield s, torch.clamp(torch.round(-half - lo / s), -half, half - 1)


def _error(x, s, z, bits, norm):
    """Σ|x̂ − x|^norm of a candidate: its fp32 differences, raised and summed in fp64."""
    half = 2 ** (bits - 1)
    d = s * (torch.clamp(torch.round(x / s) + z, -half, half - 1) - z) - x
    return d.double().abs().pow(norm).sum(1, keepdim=True)


@pytest.mark.parametrize("sym", [True, False])
@pytest.mark.parametrize("norm", [0.99, 1.0, 1.7, 2.4, 3.0, 3.01])
@pytest.mark.parametrize("rows,cols,bits,grid,shrink", [
    (64, 128, 4, 50, 0.5),      # the scripts' search
    (64, 16, 2, 50, 0.5), (64, 100, 8, 50, 0.5), (5, 6000, 4, 50, 0.5),
    (32, 128, 8, 36, 0.89),     # values up to 920 steps of the smallest scale
    (16, 1000, 3, 32, 1.0)])
def test_the_best_candidate_is_found(dev, rows, cols, bits, grid, shrink, norm, sym):
    from g2ptq_amd import WeightQuantizer
    print(f"clip search {rows}x{cols} W{bits} norm={norm} sym={sym} grid={grid}", flush=True)
    g = gen(int(100 * norm) + rows + cols)
    x = torch.randn(rows, cols, generator=g) * 0.02
    x[0, 0] = 0.3
    x[1] = x[1].abs()
    x[2] = -x[2].abs()
    x[3] = torch.round(x[3] * 200) / 64
    x = x.to(dev)
    q = WeightQuantizer()
    q.configure(bits, perchannel=True, sym=sym, mse=True, norm=norm, grid=grid, maxshrink=shrink)
    q.find_params(x)
    found = _error(x, q.scale, q.zero, bits, norm)
    least = torch.full_like(found, float("inf"))
    for s, z in _candidates(x, bits, sym, grid, int(shrink * grid)):
        least = torch.minimum(least, _error(x, s, z, bits, norm))
    # both the found and the best candidate's fp32 sums are off by at most a chain of
    # cols / 64 + 6 additions and the rounding of the power
    slack = 2 * (cols / 64 + 6 + 4) * 2.0 ** -24
    worst = ((found - least) / least.clamp_min(1e-300)).max().item()
    print(f"error above the least: {worst:.3g} of it, allowed {slack:.3g}", flush=True)
    assert torch.all(found - least <= slack * least)
