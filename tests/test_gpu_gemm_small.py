"""bta_gemm's small-tile FP64 path (32 x 32 tiles, K split over a workgroup's
waves) at the edges of its range against torch in 64 bits: the smallest K (fewer
chunks than waves), ragged chunk counts, both K-split widths, triangular ranges,
both layouts of B, a batch with strides, and C0.

Tolerance: sums of K <= 1088 products of N(0, 1) entries in any order differ by
at most ~K eps of the largest sum of magnitudes; 1e-12 of the largest entry."""
import pytest
import torch

from botorch_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("M,N,K,batch", [(64, 64, 64, 1), (64, 128, 192, 3), (192, 64, 1088, 1),
                                         (640, 640, 640, 1), (1024, 320, 320, 2)])
@pytest.mark.parametrize("kn", [False, True])
@pytest.mark.parametrize("tri", [0, _lib.GEMM_B_LOWER, _lib.GEMM_B_UPPER])
def test_small_tile_gemm(M, N, K, batch, kn, tri):
    print(f"[case] {M} {N} {K} {batch} kn={kn} tri={tri}", flush=True)
    if tri:
        K = N
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    A = torch.randn(batch, M, K, generator=g, dtype=torch.float64, device=DEV)
    B = torch.randn(batch, N, K, generator=g, dtype=torch.float64, device=DEV)  # (n, k)
    if tri == _lib.GEMM_B_LOWER:
        B = torch.tril(B)
    elif tri == _lib.GEMM_B_UPPER:
        B = torch.triu(B)
    C0 = torch.randn(batch, M, N, generator=g, dtype=torch.float64, device=DEV)
    ref = torch.stack([0.5 * (a @ b.t().contiguous()) for a, b in zip(A, B)])
    Bs = B.transpose(-1, -2).contiguous() if kn else B
    flags = tri | (_lib.GEMM_B_KN if kn else 0)
    ldb = N if kn else K
    for beta in (0.0, -2.0):
        C = torch.full((batch, M, N), float("nan"), dtype=torch.float64, device=DEV)
        _lib.check(_lib.lib().bta_gemm(
            flags, M, N, K, 0.5, _lib.ptr(A), K, _lib.ptr(Bs), ldb, beta,
            _lib.ptr(C0) if beta else None, N, _lib.ptr(C), N, batch, M * K, N * K, M * N, M * N,
            _lib.stream()), "gemm")
        want = ref + beta * C0
        assert (C - want).abs().max() < 1e-12 * want.abs().max()
