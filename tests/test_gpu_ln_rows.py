"""LayerNorm of so many rows that a wave takes one (six a CU and more), on both sides of that count: rows that fill no workgroup, widths that fill no wave, each of the
outputs, gains and activation with and without.  Reference float64; fp32 results 1e-5 of the largest value (a mean and a variance of at most 1024 values), hi/lo pairs the
same (2^-17), bf16 2^-8."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [4, 60, 256, 260, 768, 1020, 1024, 1028])
@pytest.mark.parametrize("M", [1535, 1536, 1537, 4099])
def test_forms(M, D):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    g = torch.Generator().manual_seed(M + D)
    x = (torch.randn(M, D + 4, generator=g) * 3 + 2).cuda()
    gain, shift = (torch.randn(D, generator=g).bfloat16().cuda() for _ in range(2))
    for gn, sh, act in ((gain, shift, 0), (None, None, 0), (gain, None, 1)):
        ref = torch.nn.functional.layer_norm(x[:, :D].double(), (D,), None if gn is None else gn.double(), None if sh is None else sh.double(), 1e-6)
        ref = torch.nn.functional.gelu(ref) if act else ref
        out = torch.full((M + 1, D + 4), 7.0, device="cuda")
        y = torch.full((2, M + 1, D + 8), 7.0, device="cuda", dtype=torch.bfloat16)
        for lo in ((M + 1) * (D + 8), 0):
            y.fill_(7.0)
            check(lib().mn_norm_act_split(ptr(x), D + 4, 2, ptr(gn), ptr(sh), 1e-6, act, ptr(y), D + 8, lo, ptr(out), D + 4, M, D, current_stream()), "norm")
            got = y[0, :M, :D].double() + (y[1, :M, :D].double() if lo else 0)
            assert float((out[:M, :D].double() - ref).abs().max() / ref.abs().max()) < 1e-5
            assert float((got - ref).abs().max() / ref.abs().max()) < (1e-5 if lo else 2 ** -8)
            assert bool((out[M] == 7).all()) and bool((out[:, D:] == 7).all()) and bool((y[0, M] == 7).all()) and bool((y[0, :, D:] == 7).all())
            assert lo or bool((y[1] == 7).all())
