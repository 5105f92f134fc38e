"""Every tile of the split-FP16 product (64 x 64, 128 x 64, 128 x 128, 128 x 256,
picked by size) gives each output element the same bits: the element's products are
summed in the same order whatever the tile, so a product over a larger matrix
restricted to the rows and columns of a smaller one equals the smaller product.

Sizes: one tile, ragged against the 256-column tile (N = 128 modulo 256), and both
sides of each size rule on a 256-CU chip."""
import pytest
import torch

from botorch_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _run(ah, al, bh, bl, M, N, K, flags, planes):
    C = torch.full((M, N), float("nan"), dtype=torch.float32, device=DEV)
    ch = torch.zeros(M, N, dtype=torch.float16, device=DEV) if planes else None
    cl = torch.zeros(M, N, dtype=torch.float16, device=DEV) if planes else None
    _lib.check(_lib.lib().bta_gemm_f16x3(
        flags, M, N, K, 1.0, _lib.ptr(ah), _lib.ptr(al), K, None, 1.0, _lib.ptr(bh), _lib.ptr(bl),
        K, 1.0, _lib.ptr(C), N, _lib.ptr(ch), _lib.ptr(cl), 1.0, 0, _lib.stream()), "gemm_f16x3")
    return C, ch, cl


def _planes(X):
    hi = X.half()
    return hi.contiguous(), ((X - hi.float()) * 2048).half().contiguous()


# (large M, N) per tile rule: 128 x 64, 128 x 128 (N = 128 mod 256 too), 128 x 256
@pytest.mark.parametrize("M,N", [(2048, 2048), (4096, 2048), (4096, 2176), (4096, 4096),
                                 (8192, 2176)])
def test_tiles_agree_bit_for_bit(M, N):
    print(f"[case] {M} x {N}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + N)
    A = torch.rand(M, N, generator=g, device=DEV)
    B = torch.tril(torch.randn(N, N, generator=g, device=DEV) * 0.1)
    ah, al = _planes(A)
    bh, bl = _planes(B)
    big = _run(ah, al, bh, bl, M, N, N, _lib.GEMM_B_LOWER, True)
    assert not torch.isnan(big[0]).any()
    # the same elements from 64 x 64 tiles: a few rows, and the leading columns (the
    # lower B keeps their K ranges)
    m = 128
    for r0 in (0, M - m):
        small = _run(ah[r0:r0 + m].contiguous(), al[r0:r0 + m].contiguous(), bh, bl, m, N, N,
                     _lib.GEMM_B_LOWER, True)
        for x, y in zip(big, small):
            assert torch.equal(x[r0:r0 + m], y)
    # against 64 bits: 22-bit operands, the lo x lo term dropped and FP32 sums of
    # at most 4096 products: 2e-6 of the largest entry
    ref = A[:m].double() @ B.double().t().contiguous()
    assert (big[0][:m].double() - ref).abs().max() < 2e-6 * ref.abs().max()


@pytest.mark.parametrize("M,N", [(4096, 2112), (8192, 2240), (128, 64)])
def test_odd_multiple_of_64_columns_stays_in_bounds(M, N):
    # N = 64 modulo 128 belongs to the 64-column tiles: nothing past N is written (C's
    # rows are followed by a guard row) and every entry agrees with the small product
    print(f"[case] {M} x {N}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + N)
    ah, al = _planes(torch.rand(M, N, generator=g, device=DEV))
    bh, bl = _planes(torch.tril(torch.randn(N, N, generator=g, device=DEV) * 0.1))
    C = torch.full((M + 1, N), 7.0, dtype=torch.float32, device=DEV)
    _lib.check(_lib.lib().bta_gemm_f16x3(
        _lib.GEMM_B_LOWER, M, N, N, 1.0, _lib.ptr(ah), _lib.ptr(al), N, None, 1.0, _lib.ptr(bh),
        _lib.ptr(bl), N, 1.0, _lib.ptr(C), N, None, None, 1.0, 0, _lib.stream()), "gemm_f16x3")
    assert (C[M] == 7.0).all()
    m = min(M, 128)
    small = _run(ah[M - m:].contiguous(), al[M - m:].contiguous(), bh, bl, m, N, N,
                 _lib.GEMM_B_LOWER, False)[0]
    assert torch.equal(C[M - m:M], small)


def test_upper_tiles_agree_bit_for_bit():
    M, N = 4096, 4096
    g = torch.Generator(device=DEV).manual_seed(1)
    ah, al = _planes(torch.rand(M, N, generator=g, device=DEV))
    bh, bl = _planes(torch.triu(torch.randn(N, N, generator=g, device=DEV)))
    big = _run(ah, al, bh, bl, M, N, N, _lib.GEMM_B_UPPER, False)[0]
    small = _run(ah[:128].contiguous(), al[:128].contiguous(), bh, bl, 128, N, N,
                 _lib.GEMM_B_UPPER, False)[0]
    assert torch.equal(big[:128], small)
