"""GPU: the Gram products of fp16 and fp32 activations at tile and token edges.

fp16 tokens of a plain Hessian are multiplied as fp16 (subnormals included),
fp32 tokens as the nine pairs of their bf16 planes.  A sum of T exact products
in chains of 16-token MFMA steps, split at most 16 ways and reduced in a fixed
order, is off by at most (T/16 + 16·parts)·2^-24 of Σ|x_i·x_j|, which is at most
sqrt(H_ii·H_jj).  That bound passes whole pairs over, so each pair is also
checked by itself.
"""
import pytest
import torch

from tests._util import gen

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32], ids=["fp16", "fp32"])
@pytest.mark.parametrize("C,T,size", [(1, 1, 1.0), (8, 63, 1.0), (255, 65, 1.0), (257, 1100, 1.0),
                                      (300, 5000, 1.0), (513, 2048, 1.0), (130, 700, 3e-7)])
def test_gram_of_fp16_and_fp32_tokens(dev, dtype, C, T, size):
    from g2ptq_amd import GPTQ
    print(f"gram {dtype} C={C} T={T} size={size}", flush=True)
    g = gen(C + T)
    X = (torch.randn(T, C, generator=g) * torch.exp(torch.randn(C, generator=g)) * size).to(dtype)
    lin = torch.nn.Linear(C, 4, bias=False).to(dev)
    m = GPTQ([lin])
    cut = T // 3
    for part in (X[:cut], X[cut:]):  # ragged batches, one flush
        if part.shape[0]:
            m.add_batch(0, part.to(dev), None)
    n = (1 if cut else 0) + 1
    H = m.H[0].double().cpu()
    He = X.double().t() @ X.double() * (2 / n)
    d = torch.diagonal(He).clamp_min(1e-300)
    bound = (T / 16 + 16 * 9 + 8) * 2.0 ** -24
    err = ((H - He).abs() / torch.sqrt(d.unsqueeze(0) * d.unsqueeze(1))).max().item()
    print(f"max normalized error {err:.3g}, bound {bound:.3g}", flush=True)
    assert err <= bound
    assert torch.equal(H, H.t())


@pytest.mark.parametrize("C,T,planes", [(700, 2000, 6.46e-9), (1100, 2000, 5.90e-9),
                                        (700, 8000, 5.70e-9), (2752, 14000, 3.06e-9)])
def test_fp16_products_are_no_less_exact_than_plane_pairs(dev, C, T, planes):
    """The rms distance from fp64 (of sqrt(H_ii·H_jj), over four inputs) against
    `planes`, what summing the pairs of two bf16 planes split by split gives for
    the same inputs (measured; one chain per split of theirs gave 1.2 times it)."""
    from g2ptq_amd import GPTQ
    print(f"fp16 against plane pairs C={C} T={T}", flush=True)
    off = 0.0
    for seed in range(4):
        g = torch.Generator(device=dev).manual_seed(100 * seed + C)
        X = (torch.randn(T, C, device=dev, generator=g)
             * torch.exp(torch.randn(C, device=dev, generator=g))).half()
        He = X.double().t().mm(X.double())
        d = torch.diagonal(He)
        m = GPTQ([torch.nn.Linear(C, 4, bias=False).to(dev)])
        m.add_batch(0, X.unsqueeze(0), None)
        err = (m.H[0].double() / 2 - He) / torch.sqrt(d[:, None] * d[None, :])
        off += err.pow(2).mean().item()
    rms = (off / 4) ** 0.5
    print(f"rms distance: {rms:.3g}, of the pairs {planes:.3g}", flush=True)
    assert rms <= planes


# A column that isolates plane p: its other planes change sign from token to
# token, so that over all combinations of the signs only plane p's products with
# another such column are left, 16·v_p·v_q, every term and partial sum exact (the
# result is rounded with the Hessian's factor).
# (1.5 and 1.5·2^-9 are far enough from a power of two that rounding to the
# planes returns the parts.)  16 tokens: bits 0 and 1 of the token number are
# the first group's signs, bits 2 and 3 the second's.
def _isolating_columns(dtype, shift):
    t = torch.arange(16)
    a = 1.0 - 2.0 * (t >> shift & 1)
    b = 1.0 - 2.0 * (t >> (shift + 1) & 1)
    if dtype == torch.float16:  # two planes: 8 + 3 significant bits
        values = [1.5, 1.5 * 2.0 ** -9]
        cols = [torch.full((16,), 1.5), 1.5 * a + values[1]]
    else:
        values = [1.5, 1.25 * 2.0 ** -9, 1.25 * 2.0 ** -18]
        cols = [torch.full((16,), 1.5), 1.5 * a + values[1],
                1.5 * a + 1.5 * 2.0 ** -9 * b + values[2]]
    cols = [c.to(dtype) for c in cols]
    assert all(torch.equal(c.double().to(dtype), c) for c in cols)
    return cols, values


@pytest.mark.parametrize("C", [8, 300, 16500])  # 16500: the pairs in several launches
@pytest.mark.parametrize("kind", ["gptq", "gptaq", "g2ptq"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32], ids=["fp16", "fp32"])
def test_every_pair_of_planes_counts(dev, dtype, kind, C):
    from g2ptq_amd import G2PTQ, GPTAQ, GPTQ
    print(f"plane pairs {kind} {dtype} C={C}", flush=True)
    first, values = _isolating_columns(dtype, 0)
    second, _ = _isolating_columns(dtype, 2)
    X = torch.zeros(16, C, dtype=dtype)
    for p, col in enumerate(first):
        X[:, p] = col
    at = C - len(second)  # the last columns: of another tile where C > 256
    for q, col in enumerate(second):
        X[:, at + q] = col
    X = X.to(dev)
    lin = torch.nn.Linear(C, 4, bias=False).to(dev)
    if kind == "gptq":
        m = GPTQ([lin])
    elif kind == "gptaq":
        m = GPTAQ([lin])
        fp = X.clone()
        fp[:, :len(first)] = 0  # X_fp − X = −(the first group), zero elsewhere
        m.fp_inp[0] = [fp]
    else:
        m = G2PTQ([lin], [[torch.ones(16, 1)]], [torch.ones(4, C, device=dev)], 1)
    m.add_batch(0, X.unsqueeze(0), None)
    cols = list(range(len(first))) + list(range(at, C))

    def corner(M):
        """The entries of the isolating columns, at their places."""
        M = M.reshape(C, C)
        rows = M[:, cols][cols].double().cpu()
        return {(i, j): rows[a, b] for a, i in enumerate(cols) for b, j in enumerate(cols)}
    H = corner(m.H)
    scale = {"gptq": 2.0, "gptaq": 2.0, "g2ptq": 1.0 / 16}[kind]
    # x·w and X_fp − X carry two planes, hi and lo
    rows = range(2 if kind == "g2ptq" else len(values))
    for p in rows:
        for q in range(len(values)):
            want = scale * 16 * values[p] * values[q]
            assert abs(H[p, at + q].item() - want) <= 2.0 ** -22 * want, (p, q)
            assert H[at + q, p].item() == H[p, at + q].item(), (q, p)
    if kind == "gptaq":
        D = corner(m.dXXT)
        for p in range(2):
            for q in range(len(values)):
                want = -scale * 16 * values[p] * values[q]
                assert abs(D[p, at + q].item() - want) <= -2.0 ** -22 * want, (p, q)
