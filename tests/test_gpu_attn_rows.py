"""Attention of runs of rows (attn_rows.inl) at the sizes where its grouping can go wrong: row counts around 16 / 32 / 64 vectors, several sequences
and cached tokens in one workgroup, head groups of every width, windows, chunks, tiles of pooled blocks, key splits, values inside keys.  The
reference is a plain float64 softmax; fp32 products of up to 600 terms and exponentials at 1e-6: 1e-5 of the largest value."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def run(spans, H, G, d, e, window, cap, chunk, vk, nsplit, t_max, pool=0):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    from ming_univision_amd.sequences import rows_of_spans
    L = lib()
    g = torch.Generator().manual_seed(H * 1000 + d + len(spans))
    tabs = rows_of_spans(spans, L.mn_window_attn_block_rows())
    dev = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in tabs.items() if k != "max_len"}
    M, n_seq = sum(n for _, n, _ in spans), 1 + max(s for s, _, _ in spans)
    q = torch.randn(M, H * d, generator=g) * d ** -0.5
    k = torch.randn(n_seq, t_max, G * d, generator=g)
    v = k if vk else torch.randn(n_seq, t_max, G * e, generator=g)
    n_pool = t_max // pool if pool else 1
    means = [x[:, :n_pool * pool].reshape(n_seq, n_pool, pool, -1).mean(2) for x in (k, v)] if pool else None
    ref, r = torch.empty(M, H, e, dtype=torch.float64), 0
    for s, n, past in spans:
        i, j = torch.arange(past, past + n)[:, None], torch.arange(past + n)[None]
        see = (j <= i) & ((i - j < window) if window else True) & ((i // chunk == j // chunk) if chunk else True)
        keys, vals = k[s, :past + n], v[s, :past + n]
        if pool:                                                    # the means of whole blocks before the window
            see = torch.cat([torch.arange(n_pool)[None] < (i - window + 1).clamp(min=0) // pool, see], 1)
            keys, vals = torch.cat([means[0][s], keys]), torch.cat([means[1][s], vals])
        for h in range(H):
            c = h // (H // G)
            sc = q[r:r + n].reshape(n, H, d)[:, h].double() @ keys.reshape(-1, G, d)[:, c].double().T
            sc = cap * torch.tanh(sc / cap) if cap else sc
            vv = vals.reshape(-1, G, d)[:, c, :e] if vk else vals.reshape(-1, G, e)[:, c]
            ref[r:r + n, h] = torch.softmax(sc.masked_fill(~see, -float("inf")), -1) @ vv.double()
        r += n
    kd, qd = k.cuda(), q.cuda()
    vd = kd if vk else v.cuda()
    pk, pv = [x.contiguous().cuda() for x in means] if pool else (None, None)
    n_blk, ldv = dev["blk_tab"].shape[0], G * d if vk else G * e
    ns = nsplit or L.mn_window_attn_splits(n_blk, H, G, 0, tabs["max_len"])
    ws = torch.empty(max(16, L.mn_window_attn_workspace_bytes(n_blk, H, G, e, 0, ns)), dtype=torch.uint8, device="cuda")
    out = torch.full((M + 1, H * e), 7.0, device="cuda")
    check(L.mn_window_pool_attn_blocks_gate(ptr(qd), H * d, ptr(kd), G * d, ptr(vd), ldv, ptr(pk), ptr(pv), None, cap, chunk, None, 0, ptr(dev["row_seq"]),
                                            ptr(dev["row_slot"]), ptr(dev["blk_tab"]), n_blk, 0, H, G, d, e, t_max, n_pool, window, pool, 1.0, ptr(out),
                                            H * e, None, 0, ns, ptr(ws), ws.numel(), -1, current_stream()), "attn")
    assert bool((out[M] == 7.0).all())
    err = float((out[:M].double().cpu() - ref.reshape(M, -1)).abs().max() / ref.abs().max())
    assert err < 1e-5, err


SPANS = [[(0, 1, 0)], [(0, 63, 0)], [(0, 65, 7)], [(0, 3, 0), (1, 70, 0), (2, 1, 40), (3, 17, 5)], [(1, 130, 0), (0, 5, 200)]]


@pytest.mark.parametrize("spans", SPANS)
@pytest.mark.parametrize("H,G,d,e", [(4, 1, 64, 64), (8, 2, 128, 128), (6, 6, 16, 40), (6, 3, 72, 136), (5, 1, 34, 50), (3, 1, 200, 256)])
def test_runs(spans, H, G, d, e):
    for window, cap, chunk, ns in ((0, 0.0, 0, 0), (33, 20.0, 0, 3), (0, 0.0, 48, 2), (200, 0.0, 0, 1)):
        run(spans, H, G, d, e, window, cap, chunk, False, ns, 256)


@pytest.mark.parametrize("spans", SPANS)
@pytest.mark.parametrize("H,G,d,e", [(4, 1, 64, 64), (8, 2, 128, 128), (6, 3, 72, 136), (5, 1, 34, 50)])
def test_runs_with_pooled_blocks(spans, H, G, d, e):
    """Block means before the window: tiles of means alone, of means and tokens, and rows of one tile that see different numbers of either."""
    for window, pool, ns in ((33, 4, 0), (17, 16, 1), (40, 3, 3), (1, 1, 2)):
        run(spans, H, G, d, e, window, 0.0, 0, False, ns, 256, pool)


@pytest.mark.parametrize("spans", SPANS)
@pytest.mark.parametrize("H,d,e", [(4, 64, 48), (16, 576, 512), (9, 320, 256), (2, 35, 19), (1, 200, 200), (5, 450, 442)])
def test_values_inside_keys(spans, H, d, e):
    for window, cap, chunk, ns in ((0, 0.0, 0, 0), (33, 20.0, 0, 3), (0, 0.0, 48, 2)):
        run(spans, H, 1, d, e, window, cap, chunk, True, ns, 256)


@pytest.mark.parametrize("vk", [False, True])
@pytest.mark.parametrize("H,G,d,e", [(8, 2, 128, 128), (4, 4, 64, 64), (6, 3, 72, 136), (3, 1, 200, 256), (5, 1, 34, 33), (16, 1, 576, 512)])
def test_values_that_are_not_finite(H, G, d, e, vk):
    """An infinite value at one key and a NaN at a later one: no row sees them before their keys or after they have left its window, every row between has
    them in their columns and the other columns as they are (values inside the keys: the scores are not
    finite either, and nothing of a row that sees the NaN is)."""
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    from ming_univision_amd.sequences import rows_of_spans
    if vk:
        G, e = 1, min(d, e)
    elif d > 256:
        return
    L = lib()
    T, at, nan_at = 90, 37, 40
    g = torch.Generator().manual_seed(H + d)
    tabs = rows_of_spans([(0, T, 0)], L.mn_window_attn_block_rows())
    dev = {x: torch.from_numpy(np.ascontiguousarray(y)).cuda() for x, y in tabs.items() if x != "max_len"}
    q, k = torch.randn(T, H * d, generator=g) * d ** -0.5, torch.randn(T, G, d, generator=g)
    v = k[..., :e] if vk else torch.randn(T, G, e, generator=g)
    qd, kd = q.cuda(), k.cuda()
    vd = kd if vk else v.cuda()
    vd[at, :, 1], vd[nan_at, :, 3] = float("inf"), float("nan")
    n_blk = dev["blk_tab"].shape[0]
    for window, ns in ((0, 1), (20, 1), (0, 3)):
        ws = torch.empty(max(16, L.mn_window_attn_workspace_bytes(n_blk, H, G, e, 0, ns)), dtype=torch.uint8, device="cuda")
        out = torch.empty(T, H * e, device="cuda")
        check(L.mn_window_pool_attn_blocks_gate(ptr(qd), H * d, ptr(kd), G * d, ptr(vd), G * (d if vk else e), None, None, None, 0.0, 0, None, 0, ptr(dev["row_seq"]),
                                                ptr(dev["row_slot"]), ptr(dev["blk_tab"]), n_blk, 0, H, G, d, e, T, 1, window, 0, 1.0, ptr(out), H * e,
                                                None, 0, ns, ptr(ws), ws.numel(), -1, current_stream()), "attn")
        got = out.view(T, H, e).cpu().double()
        i, j = torch.arange(T)[:, None], torch.arange(T)[None]
        see = (j <= i) & ((i - j < window) if window else True)
        for h in range(H):
            c = h // (H // G)
            p = torch.softmax((q.view(T, H, d)[:, h].double() @ k[:, c].double().T).masked_fill(~see, -float("inf")), -1)
            mine, ref = got[:, h], p @ v[:, c].double()
            if vk:
                hit = see[:, at] | see[:, nan_at]
                fin = torch.isfinite(mine)
                assert not bool(fin[see[:, nan_at]].any()) and not bool(fin[hit, 1].any()) and bool(fin[~hit].all())
                mine, ref = mine[~hit], ref[~hit]
            else:
                for col, key, odd in ((1, at, torch.isposinf), (3, nan_at, torch.isnan)):
                    assert torch.equal(odd(mine[:, col]), see[:, key]), (h, col)
                    ref[see[:, key], col], mine[see[:, key], col] = 0.0, 0.0
            assert float((mine - ref).abs().max() / ref.abs().max()) < 1e-5


@pytest.fixture
def dev_lib():
    """The same code with the switches of mingnative_dev.h, in the place of the product library."""
    import ctypes
    import os
    from ming_univision_amd import _lib
    shipped = _lib.lib()
    handle = ctypes.CDLL(os.path.join(os.path.dirname(_lib.LIB_PATH), "libmingnative_dev.so"))
    for name, (res, args) in _lib.SYMBOLS.items():
        fn = getattr(handle, name)
        fn.restype, fn.argtypes = res, args
    _lib._lib = handle
    yield handle
    handle.mn_attn_rows_tune(-1)
    _lib._lib = shipped


# sequences that end inside a group, begin inside one, fill one, and many in one; rows alone, drafted rows and prompts beside each other
MIXED = SPANS + [[(i, 16, 0) for i in range(9)], [(0, 61, 3)] + [(1 + i, 2, 30 + i) for i in range(21)] + [(30, 70, 0)], [(i, 1 + i % 5, 7 * i) for i in range(30)]]


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("H,G,d,e,vk", [(4, 1, 64, 64, 0), (8, 2, 128, 128, 0), (6, 6, 16, 40, 0), (6, 3, 72, 136, 0), (5, 1, 34, 50, 0), (3, 1, 200, 256, 0), (4, 1, 64, 48, 1),
                                        (16, 1, 576, 512, 1), (1, 1, 320, 256, 1), (2, 1, 35, 19, 1)])
def test_either_form(dev_lib, form, H, G, d, e, vk):
    """Groups of 64 (32) query vectors and runs in workgroups of their own, whatever the rule would take."""
    dev_lib.mn_attn_rows_tune(form)
    for spans in MIXED:
        for window, cap, chunk, ns, pool in ((0, 0.0, 0, 1, 0), (33, 20.0, 0, 3, 0), (0, 0.0, 48, 2, 0), (17, 0.0, 0, 1, 0 if vk else 4)):
            run(spans, H, G, d, e, window, cap, chunk, bool(vk), ns, 256, pool)
    test_values_that_are_not_finite(H, G, d, e, bool(vk))


def test_more_runs_than_the_groups_workgroups_look_at_together():
    """36000 (run, head, split) tasks of groups that hold several sequences."""
    run([(i, 1 + i % 2, 5) for i in range(600)], 20, 20, 16, 16, 0, 0.0, 0, False, 3, 16)


def test_three_splits_of_many_groups():
    """More than 256 workgroups in a head and split: every group exactly once whatever the launch order."""
    run([(0, 700, 0), (1, 700, 0), (2, 700, 0)], 5, 1, 16, 16, 0, 0.0, 0, False, 3, 704)
    run([(0, 700, 0), (1, 701, 0)], 4, 1, 32, 32, 0, 0.0, 0, True, 3, 704)


@pytest.mark.parametrize("n", [1, 16, 17, 32, 33, 300])
@pytest.mark.parametrize("H,r,e", [(4, 64, 48), (16, 128, 128), (7, 35, 19), (1, 200, 200), (20, 256, 192), (5, 442, 442), (16, 512, 448), (9, 576, 512), (3, 640, 512),
                                   (2, 700, 0), (17, 1024, 0), (1, 33, 0), (2, 130, 0), (2, 513, 0), (2, 1022, 0)])
def test_decode_rows_over_latents(n, H, r, e):
    """One row a sequence, values inside the keys: n, n + 1 and 1 keys, with and without key splits, a window and a soft cap, heads beyond 16.  e = 0:
    only mn_latent_attn takes the size."""
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    L = lib()
    g = torch.Generator().manual_seed(n + H + r)
    lens, t_max = [n, n + 1, 1], 304
    k = torch.randn(3, t_max, r, generator=g)
    q = torch.randn(3, H * r, generator=g) * r ** -0.5
    kd, qd = k.cuda(), q.cuda()
    seq, ln = torch.arange(3, dtype=torch.int32, device="cuda"), torch.tensor(lens, dtype=torch.int32, device="cuda")
    slot = ln - 1
    blk = torch.stack([seq, torch.ones_like(seq)], 1).contiguous()

    def want(cols, window=0, cap=0.0):
        out = []
        for i, m in enumerate(lens):
            first = max(0, m - window) if window else 0
            s = q[i].reshape(H, r).double() @ k[i, first:m].double().T
            s = cap * torch.tanh(s / cap) if cap else s
            out.append(torch.softmax(s, -1) @ k[i, first:m, :cols].double())
        return torch.stack(out)

    for ks in (1, 3):
        lat = torch.full((4, H, r), 7.0, device="cuda")
        ws = torch.empty(max(16, L.mn_latent_attn_workspace_bytes(3, H, r, ks)), dtype=torch.uint8, device="cuda")
        check(L.mn_latent_attn(ptr(qd), ptr(kd), ptr(seq), ptr(ln), ptr(blk), 3, 3, H, r, t_max, n + 1, ks, ptr(lat), ptr(ws), ws.numel(), current_stream()), "latent")
        ref = want(r)
        assert bool((lat[3] == 7.0).all()) and float((lat[:3].double().cpu() - ref).abs().max() / ref.abs().max()) < 1e-5
    if not e:
        return
    for window, cap, ns in ((0, 0.0, 1), (20, 5.0, 1), (0, 5.0, 3), (40, 0.0, 2)):
        ws = torch.empty(max(16, L.mn_window_attn_workspace_bytes(3, H, 1, e, 1, ns)), dtype=torch.uint8, device="cuda")
        out = torch.full((4, H * e), 7.0, device="cuda")
        check(L.mn_window_pool_attn_blocks_gate(ptr(qd), H * r, ptr(kd), r, ptr(kd), r, None, None, None, cap, 0, None, 0, ptr(seq), ptr(slot), None, 3, 1, H, 1, r, e,
                                                t_max, 1, window, 0, 1.0, ptr(out), H * e, None, 0, ns, ptr(ws), ws.numel(), -1, current_stream()), "attn")
        ref = want(e, window, cap).reshape(3, -1)
        assert bool((out[3] == 7.0).all()) and float((out[:3].double().cpu() - ref).abs().max() / ref.abs().max()) < 1e-5


@pytest.mark.parametrize("H,r,ks", [(16, 64, 1), (5, 256, 3), (20, 512, 1), (33, 35, 2)])
def test_as_many_runs_as_rows_of_uneven_length(H, r, ks):
    """Runs of three and two rows beside empty ones: the launch is cut for runs of one row."""
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    L = lib()
    g = torch.Generator().manual_seed(H + r)
    k, q = torch.randn(2, 48, r, generator=g), torch.randn(5, H * r, generator=g) * r ** -0.5
    seq, ln = torch.tensor([0, 0, 0, 1, 1], dtype=torch.int32), torch.tensor([38, 39, 40, 1, 2], dtype=torch.int32)
    blk = torch.tensor([[0, 3], [0, 0], [3, 2], [0, 0], [0, 0]], dtype=torch.int32)
    kd, qd, sd, ld, bd = k.cuda(), q.cuda(), seq.cuda(), ln.cuda(), blk.cuda()
    lat = torch.full((6, H, r), 7.0, device="cuda")
    ws = torch.empty(max(16, L.mn_latent_attn_workspace_bytes(5, H, r, ks)), dtype=torch.uint8, device="cuda")
    check(L.mn_latent_attn(ptr(qd), ptr(kd), ptr(sd), ptr(ld), ptr(bd), 5, 5, H, r, 48, 40, ks, ptr(lat), ptr(ws), ws.numel(), current_stream()), "latent")
    ref = torch.stack([torch.softmax(q[m].reshape(H, r).double() @ k[seq[m], :ln[m]].double().T, -1) @ k[seq[m], :ln[m]].double() for m in range(5)])
    assert bool((lat[5] == 7.0).all()) and float((lat[:5].double().cpu() - ref).abs().max() / ref.abs().max()) < 1e-5
