"""Row operators of latent-cache decoders in their 16-byte form and beside it: the form a call takes follows from its size, strides and pointers, and
both are the same function (oracle: the norms and the filter in 64 bits)."""
import pytest
import torch

from tests import pizitar_oracle as O

pytestmark = pytest.mark.gpu


def _bf(t):
    return t.to(torch.bfloat16)


def _err(got, want):
    return float((got.double().cpu() - want).abs().max() / want.abs().max().clamp(min=1e-30))


def _at(t, offset, ld):
    """rows of t [M, n] in a buffer `offset` floats past an aligned start, ld apart"""
    M, n = t.shape
    buf = torch.zeros(offset + M * ld + 8, device="cuda", dtype=t.dtype)
    view = buf[offset:offset + M * ld].view(M, ld)
    view[:, :n] = t.cuda()
    return view


# one value quad, less than a wave, one workgroup's edge, the largest row; an odd size, an odd stride and an odd start take the other form
@pytest.mark.parametrize("n, taps, ld, offset", [(4, 5, 4, 0), (252, 6, 256, 4), (260, 7, 260, 0), (2048, 4, 2052, 0), (4096, 8, 4096, 0), (1020, 1, 1020, 0),
                                                 (1022, 3, 1024, 0), (1024, 4, 1025, 0), (1024, 4, 1024, 1)])
def test_fused_rows(n, taps, ld, offset):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    g = torch.Generator().manual_seed(n + taps)
    M, seqs, slots = 3, [4, 0, 2], [0, 2, 9]
    wa, ba, wb, bb = (_bf(1 + 0.3 * torch.randn(n, generator=g)) for _ in range(4))
    tw = _bf(torch.randn(n, taps, generator=g))
    x, gate, y = (torch.randn(M, n, generator=g) for _ in range(3))
    past = torch.randn(5, max(taps - 1, 1), n, generator=g)
    dev = [t.cuda() for t in (wa, ba, wb, bb, tw)]
    row_seq, row_slot = (torch.tensor(v, dtype=torch.int32, device="cuda") for v in (seqs, slots))
    for gated in (False, True):
        for filt in (False, True):
            xd, gd, yd = (_at(t, offset, ld) for t in (x, gate, y))
            no, h = _at(torch.zeros(M, n), offset, ld), _at(torch.zeros(M, n), offset, ld)
            state = past.cuda().clone()
            check(lib().mn_gated_norm_filter_rows(ptr(xd), ld, ptr(gd) if gated else None, ld, ptr(yd), ld, ptr(dev[0]), ptr(dev[1]), ptr(dev[2]), ptr(dev[3]), 1e-6,
                                                  ptr(no), ld, ptr(dev[4]), taps, ptr(state), ptr(row_seq), ptr(row_slot), ptr(h) if filt else None, ld, M, n,
                                                  current_stream()))
            xr = x.double()
            if gated:
                xr = xr + O.affine_layer_norm(torch.sigmoid(gate.double()) * y.double(), wa.double(), ba.double(), 1e-6)
            nr = O.affine_layer_norm(xr, wb.double(), bb.double(), 1e-6)
            assert _err(xd[:, :n], xr) < 1e-5 and _err(no[:, :n], nr) < 1e-5
            if not filt:
                assert torch.equal(state.cpu(), past)
                continue
            for m in range(M):
                want = nr[m] + nr[m] * tw[:, taps - 1].double()
                for k in range(1, taps):
                    if slots[m] - k >= 0:
                        want = want + tw[:, taps - 1 - k].double() * past[seqs[m], k - 1].double()
                assert _err(h[m, :n], want) < 1e-5
                if taps > 1:                                         # the state moved on by this row
                    assert torch.equal(state[seqs[m], 0], no[m, :n]) and torch.equal(state[seqs[m], 1:].cpu(), past[seqs[m], :-1])


@pytest.mark.parametrize("n, ld, offset", [(4, 4, 0), (256, 256, 0), (260, 264, 4), (768, 1792, 0), (2052, 2052, 0), (4096, 4096, 0), (4100, 4100, 0), (513, 516, 0), (512, 513, 0),
                                           (512, 512, 2)])
def test_rms_rows(n, ld, offset):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    g = torch.Generator().manual_seed(n)
    M = 5
    x, w = torch.randn(M, n, generator=g), _bf(1 + 0.3 * torch.randn(n, generator=g))
    xd, wd = _at(x, offset, ld), w.cuda()
    want = O.rms_norm(x.double(), w.double(), 1e-6)
    y, y16 = torch.zeros(M, n, device="cuda"), torch.zeros(M, n, device="cuda", dtype=torch.bfloat16)
    check(lib().mn_rms_rows(ptr(xd), ld, ptr(wd), 1e-6, ptr(y), n, ptr(y16), n, None, None, 0, M, n, current_stream()))
    assert _err(y, want) < 1e-5 and torch.equal(y16, y.to(torch.bfloat16))
    arena = torch.zeros(2, M + 1, n, device="cuda")
    seq = torch.ones(M, dtype=torch.int32, device="cuda")
    slot = torch.arange(M, 0, -1, dtype=torch.int32, device="cuda")
    check(lib().mn_rms_rows(ptr(xd), ld, ptr(wd), 1e-6, ptr(arena), n, None, 0, ptr(seq), ptr(slot), M + 1, M, n, current_stream()))
    assert torch.equal(arena[1, 1:].flip(0), y) and float(arena[0].abs().max()) == 0 and float(arena[1, 0].abs().max()) == 0
