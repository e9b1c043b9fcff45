"""A stack of vision-transformer blocks as one call (mn_vit_blocks) where its routes part: rows whose residual products run split-K with the next LayerNorm in
the tail and rows that add in place, SwiGLU and GELU, hidden sizes that fill no tile of K, one and three blocks, both operand regimes.  The
reference is float64 on the same bf16 weights.  bf16 operands: some 2^-9 a product over three blocks, 2e-2 of the largest value; hi / lo: 1e-4."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def ln(x, g, b):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], g.double(), b.double(), 1e-6)


def reference(x, ws, B, T, D, hidden, gelu, causal):
    x = x.double()
    for n1g, n1b, wqkv, bqkv, wo, bo, n2g, n2b, wu, bu, wd, bd in ws:
        q, k, v = (ln(x, n1g, n1b) @ wqkv.double().T + bqkv.double()).reshape(B, T, 3, D // 64, 64).permute(2, 0, 3, 1, 4).contiguous()
        s = q @ k.transpose(-1, -2).contiguous() / 8
        s = s.masked_fill(~torch.ones(T, T, dtype=torch.bool, device=x.device).tril(), -float("inf")) if causal else s
        x = x + (torch.softmax(s, -1) @ v).transpose(1, 2).reshape(B * T, D) @ wo.double().T + bo.double()
        u = ln(x, n2g, n2b) @ wu.double().T + bu.double()
        h = torch.nn.functional.gelu(u) if gelu else torch.nn.functional.silu(u[:, :hidden]) * u[:, hidden:]
        x = x + h @ wd.double().T + bd.double()
    return x


@pytest.mark.parametrize("precise", [0, 1])
@pytest.mark.parametrize("B,T,D,depth,hidden,gelu,causal", [(1, 65, 512, 3, 512, 1, 0), (2, 33, 128, 1, 128, 0, 1), (1, 1, 64, 2, 64, 1, 1), (3, 200, 576, 2, 1536, 0, 0), (40, 257, 768, 2, 512, 0, 1),
                                                            (1, 257, 512, 2, 520, 0, 0), (2, 17, 128, 2, 40, 0, 0), (1, 90, 192, 1, 768, 1, 0)])
def test_stack(B, T, D, depth, hidden, gelu, causal, precise):
    from ming_univision_amd._lib import PP, check, current_stream, lib, ptr
    if precise and hidden % 64:
        hidden = 64 * (hidden // 64 + 1)
    g = torch.Generator().manual_seed(D + hidden + T)

    def w(*shape, std=None, mean=0.0):
        return (mean + torch.randn(*shape, generator=g) * (std or shape[-1] ** -0.5)).bfloat16().cuda()
    up = hidden if gelu else 2 * hidden
    ws = [(w(D, std=0.1, mean=1.0), w(D, std=0.1), w(3 * D, D), w(3 * D, std=0.1), w(D, D), w(D, std=0.1), w(D, std=0.1, mean=1.0), w(D, std=0.1),
           w(up, D), w(up, std=0.1), w(D, hidden), w(D, std=0.1)) for _ in range(depth)]
    fin_g, fin_b = w(D, std=0.1, mean=1.0), w(D, std=0.1)
    x = torch.randn(B * T, D, generator=g).cuda()
    ref = reference(x, ws, B, T, D, hidden, gelu, causal)
    table = (C.c_void_p * (12 * depth))(*[t.data_ptr() for b in ws for t in b])
    n = lib().mn_vit_blocks_workspace_bytes(B, T, D, hidden, gelu, precise)
    buf = torch.full((n + 256,), 77, dtype=torch.uint8, device="cuda")
    out = None if precise else torch.empty(B * T, D, dtype=torch.bfloat16, device="cuda")
    for fin_gelu in (0, 1):
        y = x.clone()
        check(lib().mn_vit_blocks(ptr(y), B, T, D, depth, C.cast(table, PP), hidden, gelu, causal, precise, 1e-6, ptr(None if precise else fin_g),
                                  ptr(None if precise else fin_b), fin_gelu, ptr(out), ptr(buf), n, current_stream()), "blocks")
        assert float((y.double() - ref).abs().max() / ref.abs().max()) < (1e-4 if precise else 2e-2)
        assert bool((buf[n:] == 77).all())
        if not precise:
            want = ln(ref, fin_g, fin_b)
            want = torch.nn.functional.gelu(want) if fin_gelu else want
            assert float((out.double() - want).abs().max() / want.abs().max()) < 3e-2
    assert lib().mn_vit_blocks(ptr(y), B, T, D, depth, C.cast(table, PP), hidden, gelu, causal, precise, 1e-6, ptr(fin_g), ptr(fin_b), 0, ptr(out), ptr(buf), n - 1,
                               current_stream()) < 0
