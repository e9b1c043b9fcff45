"""Blocks of few rows, whose products take their LayerNorm or their residual with them (mn_vit_blocks, bf16 regime): the edges of 16- and 32-row tiles, one column tile and
many, K of less than a stage, whole stages and a remainder, both activations, one row above the rule.  The reference is float64 with the kernels' own roundings (normed rows, qkv,
attention and hidden units to bf16).  What is left: attention multiplies probabilities of bf16 (2^-9 each: 1.1e-3 of its output's norm, not in the reference), which moves
roundings behind it, as fp32 sums in another order do, by as much in each of the three products that follow: 4.5e-3 of the update's norm over one block, twice that over two."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def r16(t):
    return t.float().bfloat16().double()


def norm(x, g, b):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], g.double(), b.double(), 1e-6)


def reference(x, blocks, B, T, D, hidden, gelu, causal):
    x = x.double()
    for n1g, n1b, wqkv, bqkv, wo, bo, n2g, n2b, wu, bu, wd, bd in blocks:
        qkv = r16(r16(norm(x, n1g, n1b)) @ wqkv.double().T + bqkv.double())
        q, k, v = qkv.reshape(B, T, 3, D // 64, 64).permute(2, 0, 3, 1, 4).contiguous()
        s = q @ k.transpose(-1, -2).contiguous() / 8
        s = s.masked_fill(~torch.ones(T, T, dtype=torch.bool, device=x.device).tril(), -float("inf")) if causal else s
        x = x + r16((torch.softmax(s, -1) @ v).transpose(1, 2).reshape(B * T, D)) @ wo.double().T + bo.double()
        u = r16(norm(x, n2g, n2b)) @ wu.double().T + bu.double()
        h = torch.nn.functional.gelu(u) if gelu else torch.nn.functional.silu(u[:, :hidden]) * u[:, hidden:]
        x = x + r16(h) @ wd.double().T + bd.double()
    return x


def weights(D, hidden, gelu, depth, gen):
    def w(*shape, std=None, mean=0.0):
        return (mean + torch.randn(*shape, generator=gen) * (std or shape[-1] ** -0.5)).bfloat16().cuda()
    up = hidden if gelu else 2 * hidden
    return [(w(D, std=0.1, mean=1.0), w(D, std=0.1), w(3 * D, D), w(3 * D, std=0.1), w(D, D), w(D, std=0.1), w(D, std=0.1, mean=1.0), w(D, std=0.1),
             w(up, D), w(up, std=0.1), w(D, hidden), w(D, std=0.1)) for _ in range(depth)], (w(D, std=0.1, mean=1.0), w(D, std=0.1))


def run(x, blocks, fin, B, T, D, hidden, gelu, causal):
    from ming_univision_amd._lib import PP, check, current_stream, lib, ptr
    table = (C.c_void_p * (12 * len(blocks)))(*[t.data_ptr() for b in blocks for t in b])
    n = lib().mn_vit_blocks_workspace_bytes(B, T, D, hidden, gelu, 0)
    buf, y = torch.full((n + 256,), 77, dtype=torch.uint8, device="cuda"), torch.cat([x, torch.full_like(x[:1], 5.0)])
    out = torch.empty(B * T, D, dtype=torch.bfloat16, device="cuda")
    check(lib().mn_vit_blocks(ptr(y), B, T, D, len(blocks), C.cast(table, PP), hidden, gelu, causal, 0, 1e-6, ptr(fin[0]), ptr(fin[1]), 0, ptr(out), ptr(buf), n, current_stream()), "blocks")
    assert bool((buf[n:] == 77).all()) and bool((y[B * T:] == 5).all())
    return y[:B * T], out


@pytest.mark.parametrize("B,T,D,hidden,gelu,causal", [(1, 1, 256, 64, 1, 0), (1, 15, 1024, 2752, 0, 1), (4, 4, 768, 2048, 0, 0), (1, 17, 512, 320, 1, 0), (1, 31, 1024, 4096, 1, 0), (2, 16, 256, 4096, 1, 1),
                                                      (1, 33, 768, 576, 0, 0), (1, 65, 1024, 2752, 0, 1), (1, 65, 768, 2048, 0, 0), (2, 65, 1024, 4096, 1, 0), (3, 65, 1024, 1344, 0, 0),
                                                      (1, 256, 1024, 4096, 1, 0), (4, 64, 512, 2112, 1, 0), (257, 1, 512, 2112, 1, 0)])
def test_few_rows(B, T, D, hidden, gelu, causal):
    gen = torch.Generator().manual_seed(D + hidden + T)
    blocks, fin = weights(D, hidden, gelu, 1, gen)
    x = (torch.randn(B * T, D, generator=gen) * 2 + 0.3).cuda()
    ref = reference(x, blocks, B, T, D, hidden, gelu, causal)
    y, out = run(x, blocks, fin, B, T, D, hidden, gelu, causal)
    assert float((y - ref).norm() / (ref - x).norm()) < 4.5e-3
    want = norm(ref, *fin)
    assert float((out.double() - want).norm() / want.norm()) < 6e-3          # (and its own rounding, 2^-9 at most)


def test_rows_do_not_depend_on_their_tile():
    gen = torch.Generator().manual_seed(3)
    blocks, fin = weights(768, 2048, 0, 2, gen)
    x = torch.randn(97, 768, generator=gen).cuda()
    ref = reference(x, blocks, 97, 1, 768, 2048, 0, 0)
    y, _ = run(x, blocks, fin, 97, 1, 768, 2048, 0, 0)
    one = torch.cat([run(x[i:i + 1], blocks, fin, 1, 1, 768, 2048, 0, 0)[0] for i in (0, 15, 16, 31, 32, 96)])
    pick = [0, 15, 16, 31, 32, 96]
    assert float((y - ref).norm() / (ref - x).norm()) < 9e-3
    assert float((one - ref[pick]).norm() / (ref[pick] - x[pick]).norm()) < 9e-3
