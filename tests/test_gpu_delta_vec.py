"""The gated delta rule with q and k in 16-byte loads (heads of exactly 32, 64, 128 or 256 values in rows of whole 16 bytes) and the same step without them: heads
one value short, rows whose stride or start is no multiple of 16 bytes; lengths around the four rows whose outputs meet and around the batch, more rows than the table
of sequences holds.  Reference and tolerance as in test_gpu_delta_sequences."""
import pytest
import torch

from tests.test_gpu_daberax import D, _api, _rows, delta_inputs, err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift,pad", [(0, 0), (0, 4), (0, 3), (1, 0), (2, 2)])
@pytest.mark.parametrize("H,G,d,e,lens", [(2, 1, 32, 32, [1, 2, 3, 4, 5, 31, 32, 33, 36]), (2, 2, 64, 17, [33, 1, 7]), (4, 2, 128, 16, [32, 5, 30]), (1, 1, 256, 20, [15, 16, 17, 1]),
                                          (2, 1, 31, 32, [33, 4]), (2, 2, 127, 16, [33, 3])])
def test_forms(H, G, d, e, lens, shift, pad):
    run(H, G, d, e, lens, shift, pad)


def test_beyond_the_table():
    run(1, 1, 32, 16, [2] * 1030 + [3], 0, 0)


def run(H, G, d, e, lens, shift, pad):
    check, stream, L, ptr = _api()
    g = torch.Generator().manual_seed(H + d + len(lens))
    n, M, w = len(lens), sum(lens), 2 * G * d + H * e
    past = [5 * (i % 2) for i in range(n)]
    q, k, v, beta, dec = delta_inputs(g, M, H, G, d, e)
    state = torch.randn(n, H, d, e, generator=g) * 0.3
    sd = state.cuda()
    r = _rows([(i, lens[i], past[i]) for i in range(n)])
    ld = (w + 3) // 4 * 4 + pad
    buf = torch.full((M * ld + 4,), float("nan"), device="cuda")     # what lies beside a row is no operand
    rows = buf[shift:shift + M * ld].view(M, ld)
    rows[:, :w] = torch.cat([q.reshape(M, -1), k.reshape(M, -1), v.reshape(M, -1)], 1).cuda()
    out = torch.full((M + 1, H * e), 7.0, device="cuda")
    check(L.mn_gated_delta_rows(ptr(rows), ld, ptr(D(torch.cat([beta, dec], 1))), 2 * H, M, H, G, d, e, ptr(sd), ptr(r["row_seq"]), ptr(r["row_slot"]), ptr(r["row_back"]),
                                0, ptr(out), H * e, stream()))
    assert bool((out[M] == 7.0).all())
    rep, r0 = H // G, 0
    for i in range(0, n):
        S = state[i].double() if past[i] else torch.zeros(H, d, e, dtype=torch.float64)
        ref = []
        for t in range(r0, r0 + lens[i]):
            kk, qq = k[t].double().repeat_interleave(rep, 0), q[t].double().repeat_interleave(rep, 0)
            S = dec[t].double()[:, None, None] * S
            u = beta[t].double()[:, None] * (v[t].double() - torch.einsum("hde,hd->he", S, kk))
            S = S + kk[:, :, None] * u[:, None]
            ref.append(torch.einsum("hde,hd->he", S, qq))
        if n < 20 or i in (0, 1, 1028, 1029, 1030):
            assert err(sd[i], S) < 2e-5, i
            if n < 20:
                assert err(out[r0:r0 + lens[i]].reshape(-1, H, e), torch.stack(ref)) < 2e-5, i
        r0 += lens[i]
