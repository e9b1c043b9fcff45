"""Batched fp32 products of 1 .. 9 rows (mn_gemm_f32_batched): one wave a column up to 2 rows (8 where an access would not be aligned), the fp32 matrix cores above.  Error of the
summed magnitudes against float64: trees of at most K / 64 + 6 roundings of 2^-24 a column, 1e-6 at K 514."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 3, 4, 7, 8, 9])
@pytest.mark.parametrize("N,K,B,off", [(128, 512, 4, 0), (1, 1, 1, 0), (50, 34, 3, 0), (17, 72, 2, 4), (64, 100, 5, 1), (200, 36, 20, 2), (512, 128, 16, 0)])
def test_few_rows(M, N, K, B, off):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    g = torch.Generator().manual_seed(M + N + K)
    A, W, bias, G = torch.randn(M, B * K + off, generator=g), torch.randn(B, N, K, generator=g).bfloat16(), torch.randn(N, generator=g).bfloat16(), torch.randn(M, B * N, generator=g)
    x = A[:, off:].reshape(M, B, K).double()
    ref = torch.stack([x[:, b] @ W[b].double().T for b in range(B)], 1)
    mag = torch.stack([x[:, b].abs() @ W[b].double().abs().T for b in range(B)], 1)
    Ad, Wd, bd, Gd = A.cuda(), W.cuda(), bias.cuda(), G.cuda()
    C = torch.full((M + 1, B * N), 7.0, device="cuda")
    C16 = torch.full((M + 1, B * N), 7.0, dtype=torch.bfloat16, device="cuda")
    check(lib().mn_gemm_f32_batched(Ad.data_ptr() + 4 * off, B * K + off, K, ptr(Wd), K, N * K, ptr(bd), ptr(C), B * N, N, ptr(C16), B * N, N, ptr(Gd), B * N, N, M, N, K, B, 0.5,
                                    current_stream()), "gemm")
    want = (0.5 * ref + bias.double()) * torch.sigmoid(G.double()).reshape(M, B, N)
    got = C[:M].cpu().double().reshape(M, B, N)
    assert bool((C[M] == 7.0).all()) and bool((C16[M] == 7.0).all())
    assert float(((got - want).abs() / (mag + bias.double().abs())).max()) < 1e-6
    assert torch.equal(C16[:M].cpu(), C[:M].cpu().bfloat16())
