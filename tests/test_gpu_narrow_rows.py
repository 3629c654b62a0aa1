"""GPU: the row kernels on many narrow rows.

The kernels that take four columns (or a word) per thread are as fast on rows narrower than
a workgroup as on wide ones: the same number of elements in narrow rows takes at
most three times what it takes in rows of 4096 (the parameters of a row are
re-read more often, and a row count that is no power of two leaves lanes idle;
a workgroup per row took 2 to 24 times).  The values are those of the kernels
that take one column (or word) per thread, bit for bit.
"""
import pytest
import torch

from tests._util import gen

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]

ELEMENTS = 1 << 23
WIDE = (ELEMENTS // 4096, 4096)
SLACK = 3.0


def _us(fn, n=20):
    """The least time of a call among three runs of n, in microseconds."""
    fn()
    best = float("inf")
    for _ in range(3):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(n):
            fn()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) / n * 1e3)
    return best


def _fake_quantize(dev, rows, cols, pad=0, seed=0):
    """A call on (rows, cols) values at a pitch of cols + pad, and its outputs."""
    from g2ptq_amd import _core, _lib
    g = gen(seed)
    ld = cols + pad
    x = torch.zeros(rows, ld)
    x[:, :cols] = torch.randn(rows, cols, generator=g)
    x = x.to(dev)
    s = (torch.rand(rows, generator=g) * 0.2 + 0.05).to(dev)
    z = torch.randint(-2, 3, (rows,), generator=g).float().to(dev)
    q, i = torch.empty_like(x), torch.empty_like(x)

    def call():
        _lib.call("g2ptq_fake_quantize", _core.stream(), _lib.ptr(x), rows, cols, ld, -1,
                  _lib.ptr(s), _lib.ptr(z), 1, 4, _lib.ptr(q), ld, _lib.ptr(i), ld, None)
    return call, [q[:, :cols], i[:, :cols]]


@pytest.mark.parametrize("cols", [4, 16, 32, 64])
def test_fake_quantize_time(dev, cols):
    wide = _us(_fake_quantize(dev, *WIDE)[0])
    narrow = _us(_fake_quantize(dev, ELEMENTS // cols, cols)[0])
    print(f"fake quantize, rows of {cols}: {narrow:.1f} us, of 4096: {wide:.1f} us", flush=True)
    assert narrow <= SLACK * wide


@pytest.mark.parametrize("rows,cols", [(1, 4), (255, 4), (257, 4), (129, 8), (65, 12), (1000, 20),
                                       (63, 64), (70001, 4), (31, 132), (5, 516), (3, 1020),
                                       (3, 1028)])
def test_fake_quantize_values(dev, rows, cols):
    print(f"fake quantize {rows}x{cols}", flush=True)
    outs = []
    for pad in (0, 1):  # a pitch off the 16-byte grid: one column per thread
        call, out = _fake_quantize(dev, rows, cols, pad, seed=rows + cols)
        call()
        outs.append([t.clone() for t in out])
    for a, b in zip(*outs):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))


def _pack(dev, rows, cols, bits, pad=0, seed=0):
    """A call that packs (rows, cols) codes and one group's scales per row."""
    from g2ptq_amd import _core, _lib
    g = gen(seed)
    ld, half = cols + pad, 2 ** (bits - 1)
    codes, scale = torch.zeros(rows, ld), torch.zeros(rows, ld)
    codes[:, :cols] = torch.randint(-half, half, (rows, cols), generator=g).float()
    scale[:, :cols] = torch.rand(rows, 1, generator=g)
    codes, scale = codes.to(dev), scale.to(dev)
    words = -(-cols // (32 // bits))
    packed = torch.empty(rows, words, dtype=torch.int32, device=dev)
    out = torch.empty(rows, 1, device=dev)
    flags = torch.zeros(1, dtype=torch.int32, device=dev)

    def call():
        _lib.call("g2ptq_pack_quantized", _core.stream(), _lib.ptr(codes), ld, _lib.ptr(scale), ld,
                  rows, cols, bits, cols, _lib.ptr(packed), words, _lib.ptr(out), 2, 1,
                  _lib.ptr(flags))
    return call, [packed, out, flags], scale


@pytest.mark.parametrize("bits,cols", [(8, 4), (4, 8), (4, 32), (8, 32)])
def test_pack_time(dev, bits, cols):
    wide = _us(_pack(dev, *WIDE, bits)[0])
    narrow = _us(_pack(dev, ELEMENTS // cols, cols, bits)[0])
    print(f"pack W{bits}, rows of {cols}: {narrow:.1f} us, of 4096: {wide:.1f} us", flush=True)
    assert narrow <= SLACK * wide


@pytest.mark.parametrize("rows,cols,bits", [(1, 4, 8), (257, 4, 8), (300, 8, 4), (63, 16, 2),
                                            (131, 32, 1), (1000, 24, 4), (70001, 4, 7),
                                            (9, 1032, 4), (5, 2056, 8)])
def test_pack_values(dev, rows, cols, bits):
    print(f"pack {rows}x{cols} W{bits}", flush=True)
    for spoil in (False, True):  # a scale off its group in the last row
        outs = []
        for pad in (0, 1):
            call, out, scale = _pack(dev, rows, cols, bits, pad, seed=rows + cols)
            if spoil:
                scale[rows - 1, cols - 1] += 1.0
            call()
            outs.append([t.clone() for t in out])
        for a, b in zip(*outs):
            assert torch.equal(a.view(torch.int32), b.view(torch.int32))
        assert (int(outs[0][2]) != 0) == spoil
