"""GPU: the Gram products of fp16 and fp32 activations at tile and token edges.

fp16 tokens of a plain Hessian are multiplied as fp16 (subnormals included);
fp32 tokens as the six bf16 plane pairs above 2^-23 of the product.  A sum of
T exact products in chains of 16-token MFMA steps, split at most 16 ways and
reduced in order, is off by at most (T/16 + 16·parts)·2^-24 of Σ|x_i·x_j| plus,
for fp32, 2^-22 for the pairs left out; Σ|x_i·x_j| is at most sqrt(H_ii·H_jj).
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
    bound = (T / 16 + 16 * 6 + 8) * 2.0 ** -24 + 2.0 ** -22
    err = ((H - He).abs() / torch.sqrt(d.unsqueeze(0) * d.unsqueeze(1))).max().item()
    print(f"max normalized error {err:.3g}, bound {bound:.3g}", flush=True)
    assert err <= bound
    assert torch.equal(H, H.t())


@pytest.mark.parametrize("C,T", [(700, 2000), (1100, 2000), (700, 8000), (2752, 14000)])
def test_fp16_products_are_no_less_exact_than_plane_pairs(dev, C, T):
    """GPTAQ's H of the same fp16 tokens is the sum over the pairs of two bf16
    planes; the rms distance of GPTQ's from fp64 is no larger (over four inputs,
    of sqrt(H_ii·H_jj))."""
    from g2ptq_amd import GPTAQ, GPTQ
    print(f"fp16 against plane pairs C={C} T={T}", flush=True)
    off = {"gptq": 0.0, "gptaq": 0.0}
    for seed in range(4):
        g = torch.Generator(device=dev).manual_seed(100 * seed + C)
        X = (torch.randn(T, C, device=dev, generator=g)
             * torch.exp(torch.randn(C, device=dev, generator=g))).half()
        He = X.double().t().mm(X.double())
        d = torch.diagonal(He)
        for name in off:
            lin = torch.nn.Linear(C, 4, bias=False).to(dev)
            m = GPTQ([lin]) if name == "gptq" else GPTAQ([lin])
            if name == "gptaq":
                m.fp_inp[0] = [X]
            m.add_batch(0, X.unsqueeze(0), None)
            err = (m.H[0].double() / 2 - He) / torch.sqrt(d[:, None] * d[None, :])
            off[name] += err.pow(2).mean().item()
    print(f"rms distance squared: fp16 {off['gptq']:.3g}, pairs {off['gptaq']:.3g}", flush=True)
    assert off["gptq"] <= off["gptaq"]
