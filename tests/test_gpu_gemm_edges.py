"""GPU: the fp32 GEMM's operand loads at ragged edges.

Operands sit in larger buffers whose other entries are NaN: a product may load
them (rows past M or N feed outputs that are not stored) but nothing stored may
depend on them.  K runs over whole and partial 16-k slabs and 32-k slabs and
over 4-k chunks and single elements, for every tile the dispatch picks.  Results
are held to fp64 componentwise: 4e-7 of |A|·|B| (the split's and the fp32 MFMA's
bound on the repository's products).
"""
import pytest
import torch

from tests._util import gen

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


@pytest.mark.parametrize("b_trans", [1, 0])
@pytest.mark.parametrize("M,N,K,pad", [
    (1, 1, 4, 4), (63, 65, 36, 4), (65, 64, 64, 0), (64, 130, 127, 1), (64, 64, 128, 0),
    (130, 63, 132, 4), (7, 200, 140, 4), (200, 7, 144, 8), (100, 100, 141, 3), (129, 257, 160, 0),
    (2100, 2050, 132, 4), (2100, 2052, 144, 4), (4100, 4096, 400, 4), (4100, 4100, 396, 4),
    (500, 7300, 2052, 4), (500, 7300, 2064, 0)])
def test_products_ignore_what_lies_outside(dev, M, N, K, pad, b_trans):
    from g2ptq_amd import _core, _lib
    print(f"gemm {M}x{N}x{K} pad={pad} b_trans={b_trans}", flush=True)
    g = gen(M + N + K)
    A = torch.full((M + 3, K + pad), float("nan"))
    A[:M, :K] = torch.randn(M, K, generator=g)
    if b_trans:
        Bt = torch.randn(N, K, generator=g)
        B = torch.full((N + 2, K + pad), float("nan"))
        B[:N, :K] = Bt
    else:
        Bt = torch.randn(N, K, generator=g)
        B = torch.full((K + 2, N + pad), float("nan"))
        B[:K, :N] = Bt.t()
    A, B = A.to(dev), B.to(dev)
    D = torch.full((M, N + 1), 7.0, device=dev)
    _lib.call("g2ptq_gemm_f32", _core.stream(), M, N, K, 1, _lib.ptr(A), A.stride(0), 0,
              _lib.ptr(B), B.stride(0), 0, b_trans, None, 0, 0, _lib.ptr(D), N + 1, 0, 1.0, 0.0)
    Ad, Bd = A[:M, :K].double(), Bt.to(dev).double()
    exact = Ad @ Bd.t()
    mass = Ad.abs() @ Bd.abs().t()
    err = ((D[:, :N].double() - exact).abs() / mass).max().item()
    print(f"max err / |A||B| {err:.3g}", flush=True)
    assert err <= 4e-7
    assert torch.all(D[:, N] == 7.0)


@pytest.mark.parametrize("b_trans,lda,ldb", [(1, 1 << 22, 1 << 22), (1, (1 << 22) + 1, 256),
                                             (0, 1 << 22, 1 << 23), (0, 256, 1 << 27)])
def test_rows_far_apart(dev, b_trans, lda, ldb):
    """Pitches past 32-bit offsets within a tile give the packed operands' bits."""
    from g2ptq_amd import _core, _lib
    M, N, K = 66, 68, 144
    span = 4 * (M * lda + (N if b_trans else K) * ldb)
    if torch.cuda.mem_get_info(dev)[0] < 1.25 * span:
        pytest.skip("not enough free device memory")
    print(f"gemm rows {lda} and {ldb} apart, b_trans={b_trans}", flush=True)
    g = gen(7)
    A, B = torch.randn(M, K, generator=g).to(dev), torch.randn(N, K, generator=g).to(dev)
    if not b_trans:
        B = B.t().contiguous()
    out = []
    for far in (False, True):
        if far:
            Af = torch.empty(M * lda, device=dev).as_strided((M, K), (lda, 1))
            Bf = torch.empty(B.shape[0] * ldb, device=dev).as_strided(B.shape, (ldb, 1))
            Af.copy_(A)
            Bf.copy_(B)
            A, B = Af, Bf
        D = torch.empty(M, N, device=dev)
        _lib.call("g2ptq_gemm_f32", _core.stream(), M, N, K, 1, _lib.ptr(A), A.stride(0), 0,
                  _lib.ptr(B), B.stride(0), 0, b_trans, None, 0, 0, _lib.ptr(D), N, 0, 1.0, 0.0)
        out.append(D)
    torch.cuda.synchronize()
    del A, B, Af, Bf
    torch.cuda.empty_cache()
    assert torch.equal(out[0].view(torch.int32), out[1].view(torch.int32))


@pytest.mark.parametrize("M,N,K", [(1024, 64, 2048), (64, 1024, 4096), (512, 500, 512)])
def test_small_products_with_b_given_by_rows(dev, M, N, K):
    """B given K×N, whose fragments every wave splits for itself, takes 1.25 times
    the N×K product's time where few workgroups run (1.5 with masked loads)."""
    from g2ptq_amd import _core, _lib
    A, B = torch.randn(M, K, device=dev), torch.randn(N * K, device=dev)
    D = torch.empty(M, N, device=dev)

    def us(b_trans, n=30):
        best = float("inf")
        for _ in range(4):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(n):
                _lib.call("g2ptq_gemm_f32", _core.stream(), M, N, K, 1, _lib.ptr(A), K, 0,
                          _lib.ptr(B), K if b_trans else N, 0, b_trans, None, 0, 0, _lib.ptr(D), N,
                          0, 1.0, 0.0)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) / n * 1e3)
        return best
    kn, nk = us(0), us(1)
    print(f"{M}x{N}x{K}: B by rows {kn:.1f} us, by columns {nk:.1f} us", flush=True)
    assert kn <= 1.4 * nk
