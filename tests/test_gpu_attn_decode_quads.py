"""Attention of decode rows by groups of 16 keys a wave: key counts around the groups, tiles and splits, heads of 68 .. 128 values, one to four heads a key head and twelve (in chunks), windows,
chunks, pooled blocks, a sink, a soft cap, gates and bf16 results, and the join of 2 .. 9 splits of one row.  Slots behind a row's position hold NaN: nothing of them may be read into a result.
The reference is a float64 softmax; fp32 products of up to 600 terms and exponentials at 1e-6: 1e-5 of the largest value."""
import pytest
import torch

pytestmark = pytest.mark.gpu

T = 640


@pytest.mark.parametrize("ns", [1, 2, 5, 9])
@pytest.mark.parametrize("H,G,d,e", [(16, 4, 128, 128), (3, 3, 68, 100), (4, 2, 124, 72), (12, 1, 128, 128), (6, 2, 96, 128)])
@pytest.mark.parametrize("window,pool,chunk,cap,extra", [(0, 0, 0, 0.0, False), (100, 0, 0, 5.0, True), (64, 16, 0, 0.0, False), (0, 0, 48, 0.0, True)])
def test_decode(H, G, d, e, window, pool, chunk, cap, extra, ns):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    L = lib()
    g = torch.Generator().manual_seed(H + d + window)
    pos = torch.tensor([0, 1, 15, 16, 17, 63, 64, 65, 200, 333, T - 1], dtype=torch.int32)
    M = len(pos)
    q, k, v = torch.randn(M, H * d, generator=g) * d ** -0.5, torch.randn(M, T, G * d, generator=g), torch.randn(M, T, G * e, generator=g)
    n_pool = T // pool if pool else 1
    means = [x[:, :n_pool * pool].reshape(M, n_pool, pool, -1).mean(2).contiguous() for x in (k, v)] if pool else None
    sink, gate = torch.randn(H, generator=g), torch.randn(M, H * e, generator=g)
    ref = torch.empty(M, H, e, dtype=torch.float64)
    for r, p in enumerate(pos.tolist()):
        lo = max(0, p - window + 1) if window else 0
        lo = max(lo, p - p % chunk) if chunk else lo
        keys, vals = k[r, lo:p + 1], v[r, lo:p + 1]
        if pool:
            nb = (p - window + 1) // pool if p - window + 1 >= 0 else 0
            keys, vals = torch.cat([means[0][r, :nb], keys]), torch.cat([means[1][r, :nb], vals])
        for h in range(H):
            c = h // (H // G)
            s = keys.reshape(-1, G, d)[:, c].double() @ q[r].reshape(H, d)[h].double()
            s = cap * torch.tanh(s / cap) if cap else s
            if extra:
                s = torch.cat([s, sink[h:h + 1].double()])
            ref[r, h] = torch.softmax(s, 0)[:len(vals)] @ vals.reshape(-1, G, e)[:, c].double()
        k[r, p + 1:], v[r, p + 1:] = float("nan"), float("nan")
    if extra:
        ref = ref * torch.sigmoid(gate.double()).reshape(ref.shape)
    dev = [None if t is None else t.cuda() for t in (q, k, v, means and means[0], means and means[1], sink if extra else None, gate if extra else None, torch.arange(M, dtype=torch.int32), pos)]
    out, out16 = torch.full((M + 1, H * e), 7.0, device="cuda"), torch.full((M + 1, H * e), 7.0, dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(max(16, L.mn_window_attn_workspace_bytes(M, H, G, e, 1, ns)), dtype=torch.uint8, device="cuda")
    check(L.mn_window_pool_attn_blocks_gate(ptr(dev[0]), H * d, ptr(dev[1]), G * d, ptr(dev[2]), G * e, ptr(dev[3]), ptr(dev[4]), ptr(dev[5]), cap, chunk, ptr(dev[6]), H * e, ptr(dev[7]), ptr(dev[8]),
                                            None, M, 1, H, G, d, e, T, n_pool, window, pool, 1.0, ptr(out), H * e, ptr(out16), H * e, ns, ptr(ws), ws.numel(), -1, current_stream()), "attn")
    assert bool((out[M] == 7.0).all()) and bool((out16[M] == 7.0).all())
    got = out[:M].cpu()
    assert float((got.double() - ref.reshape(M, -1)).abs().max() / ref.abs().max()) < 1e-5
    assert torch.equal(out16[:M].cpu(), got.bfloat16())
