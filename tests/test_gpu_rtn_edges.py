"""GPU: round-to-nearest and packing on 16-byte steps and off them.

The kernels that take four columns (a whole word) per thread against the ones
that take one: the same rows with the pointer or pitch moved off a 16-byte
boundary must give the same bits, for widths with remainders in every unit.
"""
import pytest
import torch

from tests._util import gen

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


def _off(t, pad):
    """A copy of t (rows, cols) whose rows start off the 16-byte grid."""
    buf = torch.zeros(t.shape[0], t.shape[1] + pad, device=t.device, dtype=t.dtype)
    buf[:, :t.shape[1]] = t
    return buf


@pytest.mark.parametrize("rows,cols,g,bits", [(1, 4, 4, 4), (3, 32, 32, 2), (70, 1056, 32, 3),
                                              (5, 4096, 128, 8), (2, 1028, -1, 4), (9, 24, 8, 16)])
def test_fake_quantize_vector_equals_scalar(dev, rows, cols, g, bits):
    from g2ptq_amd import _core, _lib
    print(f"fake quantize {rows}x{cols} g={g} W{bits}", flush=True)
    gr = gen(rows + cols)
    n = 1 if g == -1 else cols // g
    x = torch.randn(rows, cols, generator=gr).to(dev)
    x[0, 0], x[0, 1], x[0, 2] = float("nan"), float("inf"), -0.0
    s = (torch.rand(rows, n, generator=gr) * 0.2 + 0.05).to(dev)
    z = torch.randint(-2, 3, (rows, n), generator=gr).float().to(dev)
    outs = []
    for pad in (0, 1):
        xp, q, i = _off(x, pad), _off(torch.zeros_like(x), pad), _off(torch.zeros_like(x), pad)
        _lib.call("g2ptq_fake_quantize", _core.stream(), _lib.ptr(xp), rows, cols, cols + pad, g,
                  _lib.ptr(s), _lib.ptr(z), n, bits, _lib.ptr(q), cols + pad, _lib.ptr(i),
                  cols + pad, None)
        outs.append((q[:, :cols].contiguous(), i[:, :cols].contiguous()))
    for a, b in zip(*outs):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("bits", [1, 2, 3, 4, 5, 7, 8])
@pytest.mark.parametrize("rows,cols,g", [(1, 32, 32), (3, 320, 8), (67, 1056, 32), (5, 70, 7),
                                         (4, 4096, 128)])
def test_pack_vector_equals_scalar(dev, rows, cols, g, bits):
    from g2ptq_amd import _core, _lib
    print(f"pack {rows}x{cols} g={g} W{bits}", flush=True)
    gr = gen(rows * cols + bits)
    half = 2 ** (bits - 1)
    codes = torch.randint(-half, half, (rows, cols), generator=gr).float().to(dev)
    sc = torch.rand(rows, cols // g, generator=gr).to(dev)
    pf = 32 // bits
    words = -(-cols // pf)
    for spoil in (False, True):
        scale = sc.repeat_interleave(g, 1)
        if spoil and g > 1:
            scale[rows - 1, g - 1] += 1.0
        outs = []
        for pad in (0, 1):
            c, f = _off(codes, pad), _off(scale, pad)
            packed = torch.zeros(rows, words, dtype=torch.int32, device=dev)
            out = torch.zeros(rows, cols // g, device=dev)
            flags = torch.zeros(1, dtype=torch.int32, device=dev)
            _lib.call("g2ptq_pack_quantized", _core.stream(), _lib.ptr(c), cols + pad, _lib.ptr(f),
                      cols + pad, rows, cols, bits, g, _lib.ptr(packed), words, _lib.ptr(out), 2,
                      cols // g, _lib.ptr(flags))
            outs.append((packed, out, int(flags)))
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
        assert outs[0][2] == outs[1][2] and (outs[0][2] != 0) == (spoil and g > 1)
