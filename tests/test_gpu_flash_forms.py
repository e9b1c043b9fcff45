"""Flash attention of the batch and prompt passes at the edges of its forms: 64 / 128 queries and one or two key groups a workgroup (the counts of workgroups
pick the form, so heads and images are chosen to reach each), lengths around the query blocks and key tiles.  The reference is float64 on the operands the
kernels see.  hi/lo pairs carry 17 bits: products 2^-16 of |q||k| / 8, about 5 at the largest, times a softmax's sensitivity: 1e-4 of the largest value;
bf16 weights and outputs: 2^-8, 1e-2 of the largest value."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def api():
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    return check, current_stream, lib(), ptr


@pytest.mark.parametrize("hilo", [False, True])
@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("B,T,nh", [(1, 1, 2), (2, 63, 3), (3, 64, 2), (1, 65, 2), (2, 127, 4), (1, 129, 16), (1, 192, 3), (1, 640, 16), (20, 257, 4), (4, 330, 16), (2, 1025, 12), (40, 128, 16),
                                    (40, 65, 16), (1, 1025, 16)])
def test_hd64(B, T, nh, causal, hilo):
    check, stream, L, ptr = api()
    g = torch.Generator().manual_seed(T + nh)
    x = torch.randn(B, T, 3, nh, 64, generator=g).cuda()
    x = x if hilo else x.bfloat16()
    out = torch.full((B * T + 1, nh * 64), 7.0, device="cuda", dtype=x.dtype)
    if hilo:
        split = torch.zeros(2, B * T, nh * 64, device="cuda", dtype=torch.bfloat16)
        check(L.mn_attn_prefill_hd64_f32(ptr(x), ptr(out), ptr(split), B, T, nh, causal, stream()), "flash")
        assert torch.equal(split[0], out[:B * T].bfloat16())
        assert float((split[0].float() + split[1].float() - out[:B * T]).abs().max()) <= 2.0 ** -16 * float(out[:B * T].abs().max())
    else:
        check(L.mn_attn_prefill_hd64(ptr(x), ptr(out), B, T, nh, causal, stream()), "flash")
    assert bool((out[B * T] == 7.0).all())
    see = torch.ones(T, T, dtype=torch.bool, device="cuda").tril() if causal else None
    for b in sorted({0, B - 1}):
        for h in sorted({0, nh - 1}):
            q, k, v = (x[b, :, i, h].double() for i in range(3))
            s = q @ k.T / 8
            s = s.masked_fill(~see, -float("inf")) if causal else s
            ref = torch.softmax(s, -1) @ v
            got = out[b * T:(b + 1) * T, h * 64:(h + 1) * 64].double()
            assert float((got - ref).abs().max() / ref.abs().max()) < (1e-4 if hilo else 1e-2)


@pytest.mark.parametrize("hilo", [False, True])
@pytest.mark.parametrize("n_kv,spans", [(1, [(1, 0)]), (2, [(15, 0), (17, 0)]), (4, [(65, 0)]), (2, [(33, 300)]), (4, [(700, 0)]), (4, [(300, 0), (1, 0), (290, 0), (64, 0), (300, 0), (31, 0), (299, 0), (128, 0)]),
                                        (4, [(1500, 0), (1100, 0)]), (4, [(2100, 0)])])
def test_hd128(n_kv, spans, hilo):
    check, stream, L, ptr = api()
    g = torch.Generator().manual_seed(len(spans) + spans[0][0])
    longest, past = max(t for t, _ in spans), spans[0][1]
    t_max, n_q = past + longest + 3, 4 * n_kv
    M = sum(t for t, _ in spans)
    kv = torch.randn(len(spans), 2, n_kv, t_max, 128, generator=g).cuda()
    q = (torch.randn(M, n_q, 128, generator=g) * 128 ** -0.5).cuda()
    q = q if hilo else q.bfloat16()
    out = torch.full((M + 1, n_q * 128), 7.0, device="cuda", dtype=q.dtype)
    rows, r = [], 0
    for i, (t, _) in enumerate(spans):
        rows.append([len(spans) - 1 - i, r, t] + ([past] if hilo else []))
        r += t
    tab = torch.tensor(rows, dtype=torch.int32, device="cuda")
    if hilo:
        check(L.mn_flash_prefill_gqa_hd128_f32(ptr(q), ptr(kv), t_max, n_q, n_kv, ptr(tab), len(spans), longest, ptr(out), None, 0, stream()), "flash")
    else:
        check(L.mn_flash_prefill_gqa_hd128(ptr(q), ptr(kv), t_max, n_q, n_kv, past, ptr(tab), len(spans), longest, None, 0, ptr(out), stream()), "flash")
    assert bool((out[M] == 7.0).all())
    for seq, r, t, *_ in rows:
        see = torch.ones(t, past + t, dtype=torch.bool, device="cuda").tril(past)
        for h in sorted({0, n_q - 1}):
            k, v = (kv[seq, i, h // 4, :past + t] for i in range(2))
            k, v = (k, v) if hilo else (k.bfloat16(), v.bfloat16())
            s = (q[r:r + t, h].double() @ k.double().T).masked_fill(~see, -float("inf"))
            ref = torch.softmax(s, -1) @ v.double()
            got = out[r:r + t, h * 128:(h + 1) * 128].double()
            assert float((got - ref).abs().max() / ref.abs().max()) < (1e-4 if hilo else 1e-2)
