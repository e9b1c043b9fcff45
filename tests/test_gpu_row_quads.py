"""Row operators of the hybrid decoder where they go 16 bytes at a time: the gated RMS norm around the sizes where a thread's quadruples end, the head norm with its cache append at heads that
fill half a wave and less, head counts that leave its last workgroup short, and the forms that stay value by value.  The reference is float64: a row's norm is a sum of n squares, an exponential
and six roundings, 2e-6 of the value with room for the exponential's 1e-7 at |g| up to 5; bf16 results are half a bf16 step further off."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,pad", [(4, 0), (252, 4), (1024, 0), (1028, 0), (2048, 4), (2052, 0), (4096, 0), (4100, 0), (130, 0), (1024, 1)])
def test_gated_norm(n, pad):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    g = torch.Generator().manual_seed(n)
    M, ld = 5, n + pad
    x, z, w = torch.randn(M, ld, generator=g), torch.randn(M, ld, generator=g), torch.randn(n, generator=g).bfloat16()
    y, y16 = torch.full((M, ld), 7.0, device="cuda"), torch.full((M, ld), 7.0, dtype=torch.bfloat16, device="cuda")
    xd, zd, wd = x.cuda(), z.cuda(), w.cuda()
    check(lib().mn_rms_sigmoid_gate_rows(ptr(xd), ld, ptr(wd), 1e-5, ptr(zd), ld, ptr(y), ld, ptr(y16), ld, M, n, current_stream()), "gate")
    xs = x[:, :n].double()
    ref = xs / torch.sqrt((xs * xs).mean(1, keepdim=True) + 1e-5) * w.double() * torch.sigmoid(z[:, :n].double())
    got = y[:, :n].cpu().double()
    assert float(((got - ref).abs() / ref.abs().clamp(min=1e-6)).max()) < 2e-6
    assert torch.equal(y16[:, :n].cpu(), y[:, :n].cpu().bfloat16())
    assert bool((y[:, n:] == 7.0).all()) and bool((y16[:, n:] == 7.0).all())


@pytest.mark.parametrize("H,G,dim,vdim", [(16, 4, 128, 128), (5, 1, 64, 36), (3, 3, 4, 128), (2, 1, 100, 8), (4, 2, 132, 128), (4, 2, 126, 128)])
@pytest.mark.parametrize("weights", [True, False])
def test_head_norm(H, G, dim, vdim, weights):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    g = torch.Generator().manual_seed(dim)
    M, t_max, width = 7, 11, (H + G) * dim + G * vdim
    qkv = torch.randn(M, width, generator=g)
    qw, kw = (torch.randn(2, dim, generator=g).bfloat16() if weights else (None, None))
    seq, slot = torch.arange(M, dtype=torch.int32) % 3, torch.tensor([0, 3, 10, 5, 7, 9, 1], dtype=torch.int32)
    q, k, v = torch.full((M, H * dim), 7.0, device="cuda"), torch.full((3, t_max, G * dim), 7.0, device="cuda"), torch.full((3, t_max, G * vdim), 7.0, device="cuda")
    dev = [None if t is None else t.cuda() for t in (qkv, qw, kw, seq, slot)]
    check(lib().mn_head_norm_temp_append(ptr(dev[0]), width, M, H, G, dim, vdim, ptr(dev[1]), ptr(dev[2]), 1e-6, 0.25, 0.1, 4, ptr(dev[3]), ptr(dev[4]), ptr(q), H * dim, ptr(k), ptr(v),
                                         t_max, current_stream()), "head norm")
    x = qkv[:, :(H + G) * dim].reshape(M, H + G, dim).double()
    x = x / torch.sqrt((x * x).mean(2, keepdim=True) + 1e-6)
    f = 0.25 * (1 + 0.1 * torch.log(torch.floor((slot.double() + 1) / 4) + 1))
    rq, rk = x[:, :H] * (qw.double() if weights else 1) * f[:, None, None], x[:, H:] * (kw.double() if weights else 1)
    assert float((q.cpu().double().reshape(M, H, dim) - rq).abs().max()) < 2e-6 * float(rq.abs().max())
    want_k, want_v = torch.full((3, t_max, G * dim), 7.0).double(), torch.full((3, t_max, G * vdim), 7.0)
    for m in range(M):
        want_k[seq[m], slot[m]], want_v[seq[m], slot[m]] = rk[m].reshape(-1), qkv[m, (H + G) * dim:]
    assert float((k.cpu().double() - want_k).abs().max()) < 2e-6 * float(rk.abs().max()) and torch.equal(v.cpu(), want_v)
