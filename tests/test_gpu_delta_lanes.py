"""The delta rule's walk by 32 lanes a column (one long sequence) and by 16 (many): rows around the batches of 32, value columns that fill no workgroup of 8 or 16, heads below 128 state rows
and rows that are not 16-byte aligned, key heads shared by value heads, states that go on from earlier rows.  The reference is float64; a row is some 2 dim products in fp32 and the state decays, so
errors of 2^-24 a step stay within 2e-6 of the largest value."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[1], [31], [32], [33], [97], [300], [40, 3, 90], [5] * 40])
@pytest.mark.parametrize("H,G,dim,vdim,pad", [(2, 2, 128, 128, 0), (3, 1, 100, 72, 0), (4, 2, 65, 9, 1), (1, 1, 128, 17, 4)])
def test_walk(lens, H, G, dim, vdim, pad):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    g = torch.Generator().manual_seed(sum(lens) + vdim)
    M, n = sum(lens), 2 * G * dim + H * vdim
    qkv = torch.randn(M, n + pad, generator=g)
    qkv[:, :2 * G * dim] = torch.nn.functional.normalize(qkv[:, :2 * G * dim].reshape(M, 2 * G, dim), dim=2).reshape(M, -1)
    bd = torch.cat([torch.rand(M, H, generator=g), 0.5 + 0.5 * torch.rand(M, H, generator=g)], 1)
    seq = torch.cat([torch.full((k,), i, dtype=torch.int32) for i, k in enumerate(lens)])
    back = torch.cat([torch.arange(k, dtype=torch.int32) for k in lens])
    slot = back + (seq % 2) * 7                                          # every other sequence goes on from a state
    state = torch.randn(len(lens), H, dim, vdim, generator=g)
    q, k, v = qkv[:, :n].double().split([G * dim, G * dim, H * vdim], 1)
    q, k, v = q.reshape(M, G, dim).repeat_interleave(H // G, 1), k.reshape(M, G, dim).repeat_interleave(H // G, 1), v.reshape(M, H, vdim)
    ref, S, m = torch.empty(M, H, vdim, dtype=torch.float64), state.double() * (torch.arange(len(lens)) % 2)[:, None, None, None], 0
    for i, rows in enumerate(lens):
        for _ in range(rows):
            s = S[i] * bd[m, H:].double()[:, None, None]
            u = bd[m, :H].double()[:, None] * (v[m] - (s * k[m][:, :, None]).sum(1))
            S[i] = s + k[m][:, :, None] * u[:, None]
            ref[m] = (S[i] * q[m][:, :, None]).sum(1)
            m += 1
    dev = [t.cuda() for t in (qkv, bd, state, seq, slot, back)]
    out = torch.full((M + 1, H * vdim), 7.0, device="cuda")
    check(lib().mn_gated_delta_rows(ptr(dev[0]), n + pad, ptr(dev[1]), 2 * H, M, H, G, dim, vdim, ptr(dev[2]), ptr(dev[3]), ptr(dev[4]), ptr(dev[5]), 0, ptr(out), H * vdim,
                                    current_stream()), "delta")
    assert bool((out[M] == 7.0).all())
    assert float((out[:M].cpu().double().reshape(ref.shape) - ref).abs().max() / ref.abs().max()) < 2e-6
    assert float((dev[2].cpu().double() - S).abs().max() / S.abs().max()) < 2e-6
