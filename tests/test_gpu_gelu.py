"""The exact-erf GELU that every epilogue shares, against float64 (nn.GELU(), mingtok mlp.py:34-40)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _phi_tail(a):
    return 0.5 * torch.erfc(a / math.sqrt(2.0))


@pytest.mark.parametrize("span", [0.02, 1.0, 6.0, 7.0, 16.0, 40.0])
def test_gelu_against_float64(span):
    from ming_univision_amd import ops
    x = torch.cat([torch.linspace(-span, span, 65537)[:65536], torch.randn(65536, generator=torch.Generator().manual_seed(3)) * span]).reshape(64, 2048).cuda()
    y = ops.norm_act_split(x, gelu=True, want_split=False, want_f32=True)[1]
    xd, a = x.double(), x.double().abs()
    want = xd * _phi_tail(-xd)
    # the sum's rounding; the tail's: its exponent (rounded at every step of the polynomial, 2 units of 2^-24 of it), its power of two and its product; the fit
    tail = a * _phi_tail(a)
    bound = 2.0 ** -23 * want.abs() + tail * 2.0 ** -24 * (4.0 + 2.0 * (-torch.log2(_phi_tail(a).clamp_min(1e-300)))) + 2e-10
    assert ((y.double() - want).abs() <= bound).all(), float(((y.double() - want).abs() / bound).max())


def test_gelu_special_values():
    from ming_univision_amd import ops
    big = 3.0e38
    x = torch.zeros(1, 512)
    x[0, :8] = torch.tensor([math.inf, math.nan, big, -big, 20.0, -20.0, 0.0, -0.0])
    y = ops.norm_act_split(x.cuda(), gelu=True, want_split=False, want_f32=True)[1].cpu()[0]
    assert y[0] == math.inf and math.isnan(y[1]) and y[2] == x[0, 2] and y[3] == 0 and y[4] == 20 and abs(y[5]) < 1e-30 and (y[6:] == 0).all()
