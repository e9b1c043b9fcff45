"""Batched fp32 products of many tiles, whose rows are split into three bf16 parts (mn_gemm_f32_batched): K around the 64-value steps, launches of more and of fewer tiles than two a CU,
rows whose values span forty binary orders, infinities and NaN on either side.  The reference is float64; products of parts are exact, and a result is K / 32 accumulations of 32 products and
three sums, at the worst (K / 32 + 8) roundings of 2^-24 of the summed magnitudes: 1.5e-6 at K 514."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def product(A, W):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    (M, B, K), N = A.shape, W.shape[1]
    Ad, Wd, C = A.reshape(M, B * K).cuda(), W.cuda(), torch.full((M + 1, B * N), 7.0, device="cuda")
    check(lib().mn_gemm_f32_batched(ptr(Ad), B * K, K, ptr(Wd), K, N * K, None, ptr(C), B * N, N, None, 0, 0, None, 0, 0, M, N, K, B, 1.0, current_stream()), "gemm")
    assert bool((C[M] == 7.0).all())
    return C[:M].cpu().reshape(M, B, N)


@pytest.mark.parametrize("M,N,B", [(200, 130, 12), (1000, 513, 4)])                                          # 144 and 576 tiles
@pytest.mark.parametrize("K", [1, 31, 63, 64, 65, 68, 127, 128, 130, 192, 200, 514])
def test_edges_of_k(M, N, B, K):
    g = torch.Generator().manual_seed(M + K)
    A = torch.randn(M, B, K, generator=g) * torch.exp2(torch.randint(-20, 21, (M, B, K), generator=g).float())
    W = torch.randn(B, N, K, generator=g).bfloat16()
    got, x, w = product(A, W).double(), A.double(), W.double()
    for b in range(B):
        assert float(((got[:, b] - x[:, b] @ w[b].T).abs() / (x[:, b].abs() @ w[b].abs().T)).max()) < 1.5e-6


@pytest.mark.parametrize("M,N,B", [(200, 128, 20), (1000, 512, 5)])
@pytest.mark.parametrize("K", [70, 128])
def test_not_finite(M, N, B, K):
    g = torch.Generator().manual_seed(K)
    A, W = torch.randn(M, B, K, generator=g), torch.randn(B, N, K, generator=g).bfloat16()
    big = 3.4e38                                                                                             # rounds up to an infinity in bf16
    A[3, 0, 5], A[4, 0, K - 1], A[5, 1, 9], A[6, 1, 0], A[7, 2, 1] = float("inf"), -float("inf"), float("nan"), big, float("inf")
    W[0, 7, 2], W[2, 9, 3], W[2, 11, 4], W[1, 13, 6] = float("inf"), -float("inf"), float("nan"), 0.0
    A[8, 0, 2], A[9, 2, 3] = 0.0, 1.0                                                                         # an infinite weight times zero, and times a value of one part
    W[1, 20] = 0.0
    W[1, 20, 0] = 0.5
    got, want = product(A, W), torch.einsum("mbk,bnk->mbn", A.double(), W.double())
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.float().isinf())
    assert torch.equal(got[got.isinf()], want.float()[got.isinf()])
    assert float(got[6, 1, 20]) == pytest.approx(big / 2, rel=1e-6)
