"""Products of plain bf16 rows whose small tiles are taken in bands of columns (rows and weights above 3 MB): rows and columns that fill no tile, a last band narrower than the others, every
epilogue that such products have here.  The reference is float64; a chain of K fp32 sums at random signs is within sqrt(K) 2^-24 of the summed magnitudes' root, 1e-5 of the result's largest value
with room, and half a bf16 step more for bf16 results."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1300, 1096, 1536), (1409, 1032, 1600), (901, 2056, 2048), (2100, 808, 2048), (3000, 520, 4096)])
@pytest.mark.parametrize("epilogue", ["f32", "bf16", "bf16_gelu", "f32_resid", "swiglu"])
def test_bands(M, N, K, epilogue):
    from ming_univision_amd import ops
    g = torch.Generator(device="cuda").manual_seed(M + N)
    A = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    W = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    bias = torch.randn(N, device="cuda", generator=g).bfloat16()
    y = (A.cpu().double() @ W.cpu().double().T + bias.cpu().double())
    if epilogue == "swiglu":
        got, want = ops.gemm256_swiglu(A, W, bias), torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
    elif epilogue == "f32_resid":
        C = torch.randn(M, N, device="cuda", generator=g)
        want = C.cpu().double() + y
        got = ops.gemm256(A, W, bias, "f32_resid", out=C)
    else:
        got, want = ops.gemm256(A, W, bias, epilogue), (torch.nn.functional.gelu(y) if epilogue == "bf16_gelu" else y)
    err = (got.cpu().double() - want).abs()
    room = 1e-5 * want.abs().max() + (0 if got.dtype == torch.float32 else 2 ** -8 * want.abs())
    assert bool((err <= room).all()), float((err - room).max())
