"""The small-tile forms of the wide GEMM (gemm_tile.inl): edges of the 64 / 128 tiles, one K-tile up to more K-tiles than the LDS pipelines
hold, strided operands, every epilogue, plain and hi/lo rows, against float64 products of the same bf16 operands.  Tolerances: fp32 results
3e-5 of the largest value (fp32 accumulation of <= 4096 products), bf16 results one ulp (2^-8)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

# (M, N, K): each of the plain forms (64 x 64, 64 x 128, 128 x 128 once and twice per CU) and of the hi/lo ones is the choice of one of them
SHAPES = [(1, 4, 64), (63, 60, 128), (64, 64, 192), (65, 68, 256), (65, 3072, 320), (129, 132, 576), (200, 1028, 1024), (300, 3076, 512),
          (520, 2736, 1024), (1025, 1024, 1024), (1025, 3072, 256), (1409, 3200, 128), (2048, 3072, 192), (2100, 2052, 2048), (33, 32004, 64)]


def rel(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return float((a - b).abs().max() / (b.abs().max() + 1e-30))


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_forms(M, N, K):
    from ming_univision_amd import ops
    g = torch.Generator(device="cuda").manual_seed(M * 31 + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x, b = rnd(M, K), rnd(2 * N).to(torch.bfloat16)
    w = (rnd(2 * N, K) * K ** -0.5).to(torch.bfloat16)
    w1, b1 = w[:N].contiguous(), b[:N].contiguous()
    a2, a1 = ops.split_hilo(x), x.to(torch.bfloat16)
    wide = torch.zeros(M, K + 64, dtype=torch.bfloat16, device="cuda")       # rows with a stride of their own
    wide[:, :K] = a1
    for a, xr, hilo in ((a2, a2.double().sum(0), True), (a1, a1.double(), False)):
        both = xr @ w.double().T + b.double()
        ref = both[:, :N]
        lin = (lambda e, out=None: ops.gemm256(a2, w1, b1, e, out=out)) if hilo else (lambda e, out=None: ops.gemm_bf16(wide[:, :K], w1, b1, e, out=out))
        assert rel(lin("f32"), ref) < 3e-5
        acc = rnd(M, N + 4)
        base = acc.double().clone()
        lin("f32_resid", acc[:, :N]) if not hilo else ops.linear_hilo(a2, w1, b1, out=acc[:, :N], resid=True)
        assert rel(acc[:, :N], base[:, :N] + ref) < 3e-5 and torch.equal(acc[:, N:].double(), base[:, N:])
        if not hilo:
            assert rel(lin("bf16"), ref) < 2 ** -8
            assert rel(lin("bf16_gelu"), F.gelu(ref)) < 2 ** -8
        act = F.silu(both[:, :N]) * both[:, N:]
        if hilo:
            y = ops.gemm256_swiglu_split(a2, w, b)
            assert rel(y.double().sum(0), act) < 3e-5
            if K >= 256:
                assert rel(ops.gemm256_splitk(a2, w1, b1, 2).double().sum(0), ref) < 3e-5
        else:
            assert rel(ops.gemm256_swiglu(a1, w, b), act) < 2 ** -8

