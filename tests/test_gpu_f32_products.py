"""Batched fp32 products (mn_gemm_f32_batched) around the edges of their tiles: rows 9 / 32 / 33 / 64 / 65, columns and K that fill no tile, K below
a wave's share, rows that are not 16-byte aligned, every output.  The reference is float64.  Error of the summed magnitudes: at most 64 rows are summed
as trees with the rounding errors kept (8 roundings of 2^-24 and the final ones: 1e-6 with the sigmoid's and alpha's); more rows chain
K / 2 roundings at random signs, sqrt(K / 2) 2^-24 = 1e-6 at K 514, six of those at the worst of 1e5 values."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [9, 32, 33, 64, 65, 200, 1000])
@pytest.mark.parametrize("N,K,B,off", [(128, 512, 4, 0), (1, 1, 1, 0), (50, 34, 3, 0), (513, 72, 2, 0), (96, 514, 2, 0), (64, 100, 5, 1), (200, 36, 20, 2), (16, 4, 1, 0)])
def test_products(M, N, K, B, off):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    g = torch.Generator().manual_seed(M + N + K)
    A = torch.randn(M, B * K + off, generator=g)
    W = torch.randn(B, N, K, generator=g).bfloat16()
    bias = torch.randn(N, generator=g).bfloat16()
    G = torch.randn(M, B * N, generator=g)
    x = A[:, off:].reshape(M, B, K).double()
    ref = torch.stack([x[:, b] @ W[b].double().T for b in range(B)], 1)
    mag = torch.stack([x[:, b].abs() @ W[b].double().abs().T for b in range(B)], 1)
    Ad, Wd, bd, Gd = A.cuda(), W.cuda(), bias.cuda(), G.cuda()
    tol = 1e-6 if M <= 64 else 6e-6
    for full in (False, True):
        C = torch.full((M + 1, B * N), 7.0, device="cuda")
        C16 = torch.full((M + 1, B * N), 7.0, dtype=torch.bfloat16, device="cuda")
        check(lib().mn_gemm_f32_batched(Ad.data_ptr() + 4 * off, B * K + off, K, ptr(Wd), K, N * K, ptr(bd) if full else None, ptr(C), B * N, N,
                                        ptr(C16), B * N, N, ptr(Gd) if full else None, B * N, N, M, N, K, B, 0.5, current_stream()), "gemm")
        want, room = 0.5 * ref, mag
        if full:
            want = (want + bias.double()) * torch.sigmoid(G.double()).reshape(M, B, N)
            room = mag + bias.double().abs()
        got = C[:M].cpu().double().reshape(M, B, N)
        assert bool((C[M] == 7.0).all()) and bool((C16[M] == 7.0).all())
        assert float(((got - want).abs() / room).max()) < tol
        assert torch.equal(C16[:M].cpu(), C[:M].cpu().bfloat16())


@pytest.mark.parametrize("M", [16, 256])
def test_infinities(M):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    A, W = torch.ones(M, 128), torch.ones(4, 64, 128).bfloat16()
    A[1, 5], A[2, 9], A[2, 70] = float("inf"), float("inf"), -float("inf")
    C = torch.empty(M, 256, device="cuda")
    Ad, Wd = A.cuda(), W.cuda()
    check(lib().mn_gemm_f32_batched(ptr(Ad), 128, 0, ptr(Wd), 128, 64 * 128, None, ptr(C), 256, 64, None, 0, 0, None, 0, 0, M, 64, 128, 4, 1.0,
                                    current_stream()), "gemm")
    C = C.cpu()
    assert bool((C[1] == float("inf")).all()) and bool(C[2].isnan().all()) and bool((C[0] == 128).all()) and bool((C[3:] == 128).all())
