"""Batched fp32 products of many tiles over the whole range of fp32 (mn_gemm_f32_batched): rows from subnormal values to the largest, one magnitude a row, and outputs that are
taken over again, where a scaled part overflows or a weight of the tile is infinite.  The reference is float64; the bound is test_gpu_f32_split.py's, (K / 32 + 8) roundings of 2^-24 of the summed
magnitudes, (K / 8 + 12) where outputs may be taken over again, and K roundings of subnormal sums, 2^-150 each."""
import pytest
import torch

from tests.test_gpu_f32_split import product

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,B", [(200, 130, 12), (1000, 513, 4)])
@pytest.mark.parametrize("K", [31, 128, 514])
def test_rows_of_every_magnitude(M, N, B, K):
    g = torch.Generator().manual_seed(M + K)
    low = -145 + (torch.arange(M) * 264) // M                                                    # 2^-145 .. 2^118: the sums of 514 products stay below 2^128
    A = torch.ldexp(1 + torch.rand(M, B, K, generator=g), low[:, None, None].int()) * (1 - 2 * torch.randint(0, 2, (M, B, K), generator=g))
    W = torch.randn(B, N, K, generator=g).clamp(-1.5, 1.5).bfloat16()
    got, x, w = product(A, W).double(), A.double(), W.double()
    for b in range(B):
        err, mag = (got[:, b] - x[:, b] @ w[b].T).abs(), x[:, b].abs() @ w[b].abs().T
        steps = torch.where(low >= 110, K / 8 + 12, K / 32 + 8).double()[:, None]                  # (rows that may be taken over again: eight chains)
        assert bool((err <= steps * 2.0 ** -24 * mag + K * 2.0 ** -150).all()), (b, float((err / mag).max()))


def test_outputs_beside_an_infinite_weight():
    """The finite outputs of a tile that holds an infinite weight: a chain of K / 8 sums and three more."""
    g = torch.Generator().manual_seed(4)
    M, N, B, K = 200, 130, 12, 514
    A, W = torch.randn(M, B, K, generator=g), torch.randn(B, N, K, generator=g).bfloat16()
    W[:, 3, 5] = float("inf")
    got, x, w = product(A, W).double(), A.double(), W.double()
    keep = torch.arange(N) != 3
    for b in range(B):
        ref, mag = x[:, b] @ w[b, keep].T, x[:, b].abs() @ w[b, keep].abs().T
        assert float(((got[:, b][:, keep] - ref).abs() / mag).max()) < (K / 8 + 4) * 2.0 ** -24 and bool(got[:, b, 3].isinf().all())
