"""The gated delta rule over steps of many sequences (mn_gated_delta_rows): more sequences than are walked side by side, sequences that start beyond the 2048
rows looked through at a time, lengths around the four unrolled steps and the batch, one sequence alone, stored and fresh states.  The reference is the
recurrence in float64; fp32 steps of at most 60 rows with decays below 1: 2e-5 of the largest value, the bound of the other delta tests."""
import pytest
import torch

from tests.test_gpu_daberax import D, _api, _rows, delta_inputs, err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,d,e,lens", [(4, 2, 16, 16, [1 + i % 21 for i in range(210)]), (8, 4, 128, 128, [1, 2, 3, 4, 5, 31, 32, 33, 60, 1, 7, 8, 9, 16, 17, 15, 1, 1, 2, 40]),
                                          (2, 1, 64, 20, [47]), (3, 3, 30, 5, [33, 1]), (1, 1, 200, 48, [15, 16, 17, 1, 30])])
def test_many_sequences(H, G, d, e, lens):
    check, stream, L, ptr = _api()
    g = torch.Generator().manual_seed(H + d)
    n, M = len(lens), sum(lens)
    past = [5 * (i % 2) for i in range(n)]                          # every other sequence starts from its stored state
    order = [(7 * i + 3) % n if n % 7 else (n - 1 - i) for i in range(n)]
    q, k, v, beta, dec = delta_inputs(g, M, H, G, d, e)
    state = torch.randn(n, H, d, e, generator=g) * 0.3
    sd = state.cuda()
    r = _rows([(order[i], lens[i], past[i]) for i in range(n)])
    qkv = torch.cat([q.reshape(M, -1), k.reshape(M, -1), v.reshape(M, -1)], 1)
    out = torch.full((M + 1, H * e), 7.0, device="cuda")
    check(L.mn_gated_delta_rows(ptr(D(qkv)), qkv.shape[1], ptr(D(torch.cat([beta, dec], 1))), 2 * H, M, H, G, d, e, ptr(sd), ptr(r["row_seq"]), ptr(r["row_slot"]),
                                ptr(r["row_back"]), 0, ptr(out), H * e, stream()))
    assert bool((out[M] == 7.0).all())
    rep, r0 = H // G, 0
    for i in range(n):
        sl = slice(r0, r0 + lens[i])
        S = state[order[i]].double() if past[i] else torch.zeros(H, d, e, dtype=torch.float64)
        ref = []
        for t in range(r0, r0 + lens[i]):
            kk, qq = k[t].double().repeat_interleave(rep, 0), q[t].double().repeat_interleave(rep, 0)
            S = dec[t].double()[:, None, None] * S
            u = beta[t].double()[:, None] * (v[t].double() - torch.einsum("hde,hd->he", S, kk))
            S = S + kk[:, :, None] * u[:, None]
            ref.append(torch.einsum("hde,hd->he", S, qq))
        assert err(out[sl].reshape(-1, H, e), torch.stack(ref)) < 2e-5, i
        assert err(sd[order[i]], S) < 2e-5, i
        r0 += lens[i]


@pytest.mark.parametrize("H,G,d,e,n,m", [(1, 1, 8, 4, 2048, 1), (2, 1, 36, 16, 682, 3), (3, 3, 130, 20, 1023, 2), (1, 1, 8, 16, 2049, 1), (2, 2, 70, 33, 64, 32)])
def test_tables_of_sequences(H, G, d, e, n, m):
    """Up to 2048 rows the step's sequences come from one table, filled to its last entry; more rows are looked through.  Here n sequences of m rows.  A row whose
    k . q is next to nothing has a result next to nothing: the errors are held to 2e-5 of the pass's largest value, of which every sum's terms are a part."""
    check, stream, L, ptr = _api()
    g = torch.Generator().manual_seed(n + d)
    M = n * m
    q, k, v, beta, dec = delta_inputs(g, M, H, G, d, e)
    state = torch.randn(n, H, d, e, generator=g) * 0.3
    past = torch.arange(n) % 2 * 5
    sd = state.cuda()
    r = _rows([(n - 1 - i, m, int(past[i])) for i in range(n)])
    qkv = torch.cat([q.reshape(M, -1), k.reshape(M, -1), v.reshape(M, -1)], 1)
    out = torch.full((M + 1, H * e), 7.0, device="cuda")
    check(L.mn_gated_delta_rows(ptr(D(qkv)), qkv.shape[1], ptr(D(torch.cat([beta, dec], 1))), 2 * H, M, H, G, d, e, ptr(sd), ptr(r["row_seq"]), ptr(r["row_slot"]),
                                ptr(r["row_back"]), 0, ptr(out), H * e, stream()))
    assert bool((out[M] == 7.0).all())
    S = state.flip(0).double() * (past > 0).double()[:, None, None, None]
    ref = torch.empty(n, m, H, e, dtype=torch.float64)
    rows = lambda t, w: t.double().reshape(n, m, *w)  # noqa: E731
    qq, kk = (rows(t, (G, d)).repeat_interleave(H // G, 2) for t in (q, k))
    vv, bb, dd = rows(v, (H, e)), rows(beta, (H,)), rows(dec, (H,))
    for t in range(m):
        S = dd[:, t, :, None, None] * S
        u = bb[:, t, :, None] * (vv[:, t] - (S * kk[:, t, :, :, None]).sum(2))
        S = S + kk[:, t, :, :, None] * u[:, :, None]
        ref[:, t] = (S * qq[:, t, :, :, None]).sum(2)
    assert err(out[:M].reshape(n, m, H, e), ref) < 2e-5 and err(sd.flip(0), S) < 2e-5
