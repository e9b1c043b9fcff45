"""Products of 17 .. 32 rows whose workgroups take 16 rows each: row counts at the edges of the second half, columns that fill no tile, K that fills no wave's piece, gated units and every epilogue
that reads other rows, a residual updated in place.  The reference is float64; rows enter with 24 bits and sums keep their roundings: 1e-6 of the summed magnitudes with the epilogues' exponentials."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [17, 23, 24, 25, 31, 32])
@pytest.mark.parametrize("N,K,prologue,epilogue", [(2048, 2048, "none", "none"), (100, 72, "silu", "none"), (1000, 1000, "none", "resid"), (33, 520, "none", "gelu"), (1024, 512, "none", "swiglu"),
                                                   (2048, 3072, "none", "resid"), (1003, 512, "silu", "geglu_tanh"), (7, 1024, "none", "swiglu")])
def test_halves(M, N, K, prologue, epilogue, monkeypatch):
    from ming_univision_amd import ops
    real = torch.empty
    g = torch.Generator().manual_seed(M * 31 + N + K)
    pair = epilogue in ("swiglu", "geglu_tanh")
    x, w = torch.randn(M, K, generator=g), (torch.randn(N * (2 if pair else 1), K, generator=g) * K ** -0.5).bfloat16()
    b, res = torch.randn(w.shape[0], generator=g).bfloat16(), torch.randn(M, N, generator=g)
    a = torch.nn.functional.silu(x.double()) if prologue == "silu" else x.double()
    y, mag = a @ w.double().T + b.double(), a.abs() @ w.double().abs().T + b.double().abs()
    if epilogue == "swiglu":
        y, mag = torch.nn.functional.silu(y[:, :N]) * y[:, N:], mag[:, :N] * mag[:, N:]
    elif epilogue == "geglu_tanh":
        y, mag = torch.nn.functional.gelu(y[:, :N], approximate="tanh") * y[:, N:], mag[:, :N] * mag[:, N:]
    elif epilogue == "gelu":
        y = torch.nn.functional.gelu(y)
    elif epilogue == "resid":
        y, mag = y + res.double(), mag + res.double().abs()
    out = torch.full((M + 1, N), 7.0, device="cuda")
    if epilogue == "resid":
        out[:M] = res.cuda()
    scratch = []
    monkeypatch.setattr(ops.torch, "empty", lambda *a, **kw: scratch.append(real(*a, **kw).fill_(77)) or scratch[-1])
    ops.skinny_gemm(x.cuda(), w.cuda(), b.cuda(), prologue=prologue, epilogue=epilogue, out=out[:M], res=out[:M] if epilogue == "resid" else None)
    monkeypatch.undo()
    assert len(scratch) == 1 and bool((scratch[0] == 77).all())            # one launch: three would leave the rows' parts in the scratch
    assert bool((out[M] == 7.0).all())
    assert float(((out[:M].cpu().double() - y).abs() / mag).max()) < 1e-6
