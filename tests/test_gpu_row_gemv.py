"""A product of one row whose weights are one round trip (mn_skinny_gemm, one row of bf16 weights) against float64: partial and single chunks of 512 values, rows that do not
fill the waves, every prologue and epilogue it takes, an output over the row (another kernel's)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(N, K, pro, epi, seed, bias=True):
    g = torch.Generator().manual_seed(seed)
    sw = 2 if epi in ("swiglu", "geglu_tanh") else 1
    w = (torch.randn(N * sw, K, generator=g) * K ** -0.5).to(torch.bfloat16)
    b = (torch.randn(N * sw, generator=g) * 0.1).to(torch.bfloat16) if bias else None
    x, res, gate = torch.randn(1, K, generator=g) * 2 + 0.3, torch.randn(1, N, generator=g), torch.randn(1, N, generator=g)
    lg, lb = (1 + 0.2 * torch.randn(K, generator=g)).to(torch.bfloat16), (0.2 * torch.randn(K, generator=g)).to(torch.bfloat16)
    xd = x.double()
    if pro == "silu":
        xd = torch.nn.functional.silu(xd)
    elif pro == "rmsnorm":
        xd = xd / torch.sqrt((xd * xd).mean() + 1e-6) * lg.double()
    elif pro == "ln":
        c = xd - xd.mean()
        xd = c / torch.sqrt((c * c).mean() + 1e-6) * lg.double() + lb.double()
    y = xd @ w.double().T + (b.double() if bias else 0.0)
    F = torch.nn.functional
    y = dict(none=lambda: y, silu=lambda: F.silu(y), gelu=lambda: F.gelu(y), swiglu=lambda: F.silu(y[:, :N]) * y[:, N:], geglu_tanh=lambda: F.gelu(y[:, :N], approximate="tanh") * y[:, N:],
             resid=lambda: res.double() + y, resid_gate=lambda: res.double() + gate.double() * y)[epi]()
    kw = dict(prologue=pro, epilogue=epi, eps=1e-6)
    if pro in ("rmsnorm", "ln"):
        kw["ln_g"] = lg.cuda()
    if pro == "ln":
        kw["ln_b"] = lb.cuda()
    if epi.startswith("resid"):
        kw["res"] = res.cuda()
    if epi == "resid_gate":
        kw["gate"] = gate.cuda()
    kw["terms"] = xd.abs() @ w.double().abs().T
    return x.cuda(), w.cuda(), None if b is None else b.cuda(), kw, y


def _err(got, want):
    return float((got.double().cpu() - want).abs().max() / want.abs().max())


# sums of K products in 64 chains of K / 64 and a tree of six: each rounding is 2^-24 of at most the terms' sum; the bias and, behind a norm, four roundings of every value
@pytest.mark.parametrize("K", [8, 504, 512, 520, 1000, 1024, 1536, 2048, 2736, 3080, 4096])
@pytest.mark.parametrize("N", [1, 5, 1024, 1027, 3072, 4100])
def test_shapes(N, K):
    from ming_univision_amd import ops
    for pro in ("none", "rmsnorm", "ln"):
        x, w, b, kw, want = _case(N, K, pro, "none", N + K)
        terms = kw.pop("terms")
        out = torch.full((1, N + 8), 7.0, device="cuda")
        ops.skinny_gemm(x, w, b, out=out[:, :N], **kw)
        assert bool(((out[:, :N].double().cpu() - want).abs() <= 2.0 ** -24 * ((K // 64 + 12) * terms + 2 * want.abs())).all()), pro
        assert bool((out[:, N:] == 7.0).all())


@pytest.mark.parametrize("epi", ["none", "silu", "gelu", "swiglu", "geglu_tanh", "resid", "resid_gate"])
@pytest.mark.parametrize("pro", ["none", "silu", "rmsnorm", "ln"])
def test_prologues_and_epilogues(pro, epi):
    from ming_univision_amd import ops
    for N, K, bias in ((2736, 1024, True), (1500, 640, False), (2050, 2048, True)):
        x, w, b, kw, want = _case(N, K, pro, epi, N, bias)
        kw.pop("terms")
        assert _err(ops.skinny_gemm(x, w, b, **kw), want) < 2e-6


def test_output_over_the_row_and_residual_in_place():
    from ming_univision_amd import ops
    x, w, b, kw, want = _case(1024, 1024, "rmsnorm", "none", 3)
    kw.pop("terms")
    row = torch.cat([x, torch.zeros_like(x)], 1)
    one = ops.skinny_gemm(row[:, :1024], w[:8], b[:8], out=row[:, 4:12], **kw)      # (a workgroup's worth of results over the row that it reads)
    assert _err(one, want[:, :8]) < 2e-6
    x, w, b, kw, want = _case(1024, 2736, "none", "resid", 4)
    kw.pop("terms")
    h = kw["res"].clone()
    kw["res"] = h
    ops.skinny_gemm(x, w, b, out=h, **kw)
    assert _err(h, want) < 1e-6
