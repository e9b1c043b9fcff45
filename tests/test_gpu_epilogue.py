"""Epilogues of the wide products whose bf16 rows are of whole 16 bytes, and rows that are not: a length, a stride or a first column that is only a multiple of 4
keeps the 8-byte stores.  Every tile form, with and without a bias; nothing beside the result is written.  The reference is the float64 product of the same operands: one
ulp of bf16, 2^-8 of the largest value (hi/lo pairs and fp32 sums: 3e-5, as in test_gpu_gemm_tile)."""
import pytest
import torch
import torch.nn.functional as F

from tests import test_gpu_gemm_tile as G

pytestmark = pytest.mark.gpu
dev_lib = G.dev_lib


@pytest.mark.parametrize("N,pad,first", [(8, 0, 0), (64, 8, 8), (72, 4, 0), (120, 8, 4), (124, 8, 0), (136, 0, 0), (260, 4, 4), (264, 16, 8)])
@pytest.mark.parametrize("form", [0, 1, 2, 3, 4, -1])
def test_rows(dev_lib, form, N, pad, first):
    from ming_univision_amd import ops
    dev_lib.mn_gemm_tile_tune(form)
    g = torch.Generator(device="cuda").manual_seed(N + pad)
    for M, K, bias in ((1, 64, True), (67, 128, True), (130, 192, False), (257, 64, True)):
        a = torch.randn(M, K, generator=g, device="cuda").bfloat16()
        w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
        b = torch.randn(N, generator=g, device="cuda").bfloat16() if bias else None
        ref = a.double() @ w.double().T + (b.double() if bias else 0)
        for epi, want in (("bf16", ref), ("bf16_gelu", F.gelu(ref)), ("f32", ref), ("f32_resid", 2 + ref)):
            buf = torch.full((M, N + pad + first), 2.0, device="cuda", dtype=torch.bfloat16 if epi.startswith("bf16") else torch.float32)
            ops.gemm_bf16(a, w, b, epi, out=buf[:, first:first + N])
            assert G.rel(buf[:, first:first + N], want) < (2 ** -8 if epi.startswith("bf16") else 3e-5), (epi, M, K)
            assert bool((buf[:, :first] == 2).all()) and bool((buf[:, first + N:] == 2).all())


@pytest.mark.parametrize("M,N", [(1, 8), (31, 40), (47, 56), (70, 64), (130, 136), (300, 264), (300, 268)])
def test_hilo_pairs(M, N):
    from ming_univision_amd import ops
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x, b = torch.randn(M, 128, generator=g, device="cuda"), torch.randn(2 * N, generator=g, device="cuda").bfloat16()
    w = (torch.randn(2 * N, 128, generator=g, device="cuda") * 128 ** -0.5).bfloat16()
    a = ops.split_hilo(x)
    both = a.double().sum(0) @ w.double().T + b.double()
    assert G.rel(ops.gemm256_swiglu_split(a, w, b).double().sum(0), F.silu(both[:, :N]) * both[:, N:]) < 3e-5
