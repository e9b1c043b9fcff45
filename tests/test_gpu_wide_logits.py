"""hi/lo products with a matrix of 256 MB and more (a vocabulary's logits), one row tile: rows on both sides of the forms' lines, columns that fill their rounds, that do not, and that end
inside a tile, against float64 on sampled columns.  The sum of K products (hi and lo) in fp32: 2^-24 of the summed magnitudes each."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(130004, 1088), (66004, 2048), (30004, 4544)])
def test_rows(N, K):
    from ming_univision_amd import _lib
    from ming_univision_amd._lib import ptr
    L = _lib.lib()
    assert N * K * 2 >= 1 << 28
    g = torch.Generator(device="cuda").manual_seed(N)
    W = torch.empty(N, K, dtype=torch.bfloat16, device="cuda").normal_(0, K ** -0.5, generator=g)
    b = torch.randn(N, device="cuda", generator=g).bfloat16()
    cols = torch.cat([torch.arange(160, device="cuda"), torch.randint(0, N, (600,), device="cuda", generator=g), torch.arange(N - 300, N, device="cuda")])
    for M in (1, 16, 17, 32, 33, 64):
        x = torch.randn(M, K, device="cuda", generator=g)
        A = torch.empty(2, M, K, dtype=torch.bfloat16, device="cuda")
        A[0] = x
        A[1] = x - A[0].float()
        a64, w64 = A[0].double() + A[1].double(), W[cols].double()
        C = torch.full((M + 1, N), 7.0, device="cuda")
        assert L.mn_gemm256(ptr(A), K, M * K, ptr(W), K, ptr(b), ptr(C), N, M, N, K, 2, torch.cuda.current_stream().cuda_stream) == 0
        ref, mag = a64 @ w64.t() + b[cols].double(), a64.abs() @ w64.abs().t() + b[cols].double().abs()
        assert bool(((C[:M, cols].double() - ref).abs() <= (2 * K + 16) * 2.0 ** -24 * mag).all())
        assert bool((C[M] == 7.0).all()) and bool(torch.isfinite(C).all())
