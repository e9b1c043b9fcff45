"""Decode attention that appends the new key itself and splits a row's keys over workgroups, the last of which joins them (decoder steps of rows of distinct sequences), against
the launches that steps without that promise take: rows of one key, at the edges of a batch of keys and of the first split, up to the cache's end; row counts from one row to more than
a workgroup a CU; one to four query heads a key head of 64 and of 128; holes in the mask and a row that attends nothing; one long row among short ones (splits by the rows' lengths up to 128
rows, of 1024 keys above).  Both sum fp32 products of at most 9000 keys in
another order (1e-6 of the largest value), two layers and the products between them pass it on: 2e-5 of a row's norm.  And the launch by itself against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

EDGES = (0, 1, 31, 62, 63, 64, 94, 95, 96, 97, 127, 128, 129, 190, 191, 192, 200, 255, 256, 257, 383, 384, 385)


def decoder(n_q, n_kv, hd, t_max, n_seq):
    from ming_univision_amd import configuration as C
    from ming_univision_amd.bailing_moe import BailingMoeDecoder
    from ming_univision_amd.synth import synth_state_dict
    cfg = C.BailingMoeConfig(vocab_size=64, hidden_size=256, num_hidden_layers=2, num_attention_heads=n_q, num_key_value_heads=n_kv, num_experts=4, num_experts_per_tok=4,
                             num_shared_experts=1, moe_intermediate_size=64, head_dim=hd, use_bias=False, image_patch_token=60, image_start_token=61)
    sd = {k: v.to("cuda", torch.bfloat16) for k, v in synth_state_dict(C.llm_param_shapes(cfg), 5).items()}
    return BailingMoeDecoder.from_state_dict(cfg, sd, t_max=t_max, n_seq=n_seq)


def positions(M, t_max, g):
    at = [p for p in EDGES if p < t_max] + [t_max - 1]
    return torch.tensor([at[i % len(at)] if i % 3 else int(torch.randint(0, t_max, (1,), generator=g)) for i in range(1, M + 1)], dtype=torch.int32)


@pytest.mark.parametrize("n_q,n_kv,hd", [(4, 1, 128), (8, 2, 128), (4, 2, 128), (2, 2, 128), (4, 1, 64), (4, 2, 64), (4, 4, 64)])
@pytest.mark.parametrize("M,t_max,use_mask", [(1, 70, False), (1, 1400, True), (3, 400, False), (24, 1400, False), (40, 300, True), (64, 129, False), (65, 400, True), (300, 130, False)])
def test_against_separate_launches(M, t_max, use_mask, n_q, n_kv, hd):
    dec = decoder(n_q, n_kv, hd, t_max, M)
    g = torch.Generator().manual_seed(M + t_max + hd)
    past = torch.randn(dec.kv_cache.shape, generator=g).cuda()
    for turn in range(2):
        x = torch.randn(M, 256, generator=g).cuda()
        slot = positions(M, t_max, g) if turn == 0 else torch.full((M,), t_max - 1, dtype=torch.int32)
        mask = None
        if use_mask:
            mask = (torch.rand(M, t_max, generator=g) < 0.6).to(torch.uint8)
            mask[torch.arange(M), slot.long()] = 1
            if M > 1:
                mask[1] = 0                              # attends nothing: the mean of its values
            mask = mask.cuda()
        slot, seq = slot.cuda(), torch.randperm(M, generator=g).to(torch.int32).cuda()

        def step(distinct):
            dec.kv_cache.copy_(past)
            return dec.step(x, seq, slot, slot, slot + 1, key_mask=mask, distinct_sequences=distinct).clone(), dec.kv_cache.clone()
        (want, kv0), (got, kv1), (again, _) = step(False), step(True), step(True)
        assert torch.equal(got, again)
        assert float(((got - want).norm(dim=1) / want.norm(dim=1)).max()) < 2e-5
        assert float((kv1 - kv0).abs().max()) < 2e-5 * float(past.abs().max())


@pytest.mark.parametrize("n_q,n_kv,hd", [(4, 1, 128), (8, 2, 128), (4, 4, 64)])
@pytest.mark.parametrize("M,t_max,long", [(2, 9000, 8999), (5, 9000, 9000), (36, 3000, 2900), (64, 1100, 1100), (65, 2500, 2500), (127, 1200, 1000), (128, 2049, 2049), (129, 2500, 2500), (200, 1537, 1537)])
def test_one_long_row(M, t_max, long, n_q, n_kv, hd):
    dec = decoder(n_q, n_kv, hd, t_max, M)
    g = torch.Generator(device="cuda").manual_seed(M + t_max + hd)
    past = torch.randn(dec.kv_cache.shape, generator=g, device="cuda")
    x = torch.randn(M, 256, generator=g, device="cuda")
    for turn in range(3):                                # the long row first, last and in between; the others from one key to 99, the second time all but one of a single key
        slot = torch.randint(0, 99 if turn != 1 else 1, (M,), generator=g, device="cuda", dtype=torch.int32)
        slot[(0, M - 1, M // 3)[turn]] = long - 1
        seq = torch.randperm(M, generator=g, device="cuda").to(torch.int32)

        def step(distinct):
            dec.kv_cache.copy_(past)
            return dec.step(x, seq, slot, slot, slot + 1, distinct_sequences=distinct).clone()
        want, got, again = step(False), step(True), step(True)
        assert torch.equal(got, again)
        assert float(((got - want).norm(dim=1) / want.norm(dim=1)).max()) < 2e-5


@pytest.mark.parametrize("M,t_max", [(1, 64), (3, 400), (24, 1100), (65, 96), (130, 1600)])
def test_new_key_behind_a_full_cache(M, t_max):
    """A slot of t_max is written nowhere and no line of the cache behind its last is read: the step attends the cache and the new key, as one whose cache has room for it does."""
    dec, room = decoder(8, 2, 128, t_max, M), decoder(8, 2, 128, t_max + 1, M)
    g = torch.Generator(device="cuda").manual_seed(M + t_max)
    past = torch.randn(room.kv_cache.shape, generator=g, device="cuda")
    x = torch.randn(M, 256, generator=g, device="cuda")
    slot = torch.full((M,), t_max, device="cuda", dtype=torch.int32)
    slot[:M // 2] = t_max // 2
    seq, pos = torch.arange(M, device="cuda", dtype=torch.int32), slot.clamp(max=t_max - 1)
    room.kv_cache.copy_(past)
    want = room.step(x, seq, slot, pos, slot + 1, distinct_sequences=True)
    dec.kv_cache.copy_(past[..., :t_max, :])
    got = dec.step(x, seq, slot, pos, slot + 1, distinct_sequences=True)
    assert float(((got - want).norm(dim=1) / want.norm(dim=1)).max()) < 2e-5
    assert torch.equal(dec.kv_cache[:, M // 2:], past[:, M // 2:, ..., :t_max, :])
    for width in (t_max + 1, t_max):                     # a mask that covers the key behind the cache says of it too; one of the cache's length leaves it attended
        masked, seen = (torch.ones(M, n, dtype=torch.uint8, device="cuda") for n in (width, t_max + 1))
        masked[:, t_max // 3] = 0
        masked[M // 2::2, t_max:] = 0
        seen[:, :width] = masked
        room.kv_cache.copy_(past)
        want = room.step(x, seq, slot, pos, slot + 1, key_mask=seen, distinct_sequences=True)
        dec.kv_cache.copy_(past[..., :t_max, :])
        got = dec.step(x, seq, slot, pos, slot + 1, key_mask=masked, distinct_sequences=True)
        assert float(((got - want).norm(dim=1) / want.norm(dim=1)).max()) < 2e-5


def internal():
    import ctypes
    import os
    from ming_univision_amd import _lib
    dev = ctypes.CDLL(os.path.join(os.path.dirname(_lib.LIB_PATH), "libmingnative_dev.so"))
    i, l, f, p = ctypes.c_int, ctypes.c_int64, ctypes.c_float, ctypes.c_void_p
    dev.mn_attn_arrivals.restype, dev.mn_attn_arrivals.argtypes = p, [i, i, i, i, l, p, ctypes.c_size_t, p]
    dev.mn_attn_decode_fused.restype, dev.mn_attn_decode_fused.argtypes = i, [p, l, i, l, i, i, i, i, i, p, p, p, p, p, i, i, f, p, l, p, p, l, p, p, p, p, p]
    return dev


@pytest.mark.parametrize("n_q,n_kv,hd", [(8, 2, 128), (2, 1, 128), (4, 4, 64), (4, 1, 64)])
@pytest.mark.parametrize("M,t_max,use_mask", [(1, 9000, False), (3, 400, True), (24, 1400, False), (65, 2500, True), (128, 1100, False), (150, 2500, False)])
def test_against_float64(M, t_max, use_mask, n_q, n_kv, hd):
    """The launch by itself, projections in three slabs, one long row among short ones.  Fp32: a score sums hd products whose magnitudes sum to about 0.64 sqrt(hd) in some twenty roundings (7e-6 at the
    most, weights err twice that), values in chains of at most 9000 / 32: 3e-5 of a row's largest value."""
    import ctypes
    from ming_univision_amd._lib import lib, ptr
    dev, half, nz, n = internal(), hd // 2, 3, ctypes.c_int()
    g = torch.Generator(device="cuda").manual_seed(M + t_max + hd + n_q)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    kv, qkv, angle = rnd(M, 2, n_kv, t_max, hd), rnd(nz, M, n_q + 2 * n_kv, hd), 6.28 * torch.rand(t_max, half, generator=g, device="cuda")
    cos, sin, seq = angle.cos(), angle.sin(), torch.randperm(M, generator=g, device="cuda").int()
    slot = torch.randint(0, min(t_max, 300), (M,), generator=g, device="cuda").int()
    slot[M // 2] = t_max - 1
    length = slot + 1
    mask = (torch.rand(M, t_max, generator=g, device="cuda") < 0.6).to(torch.uint8) if use_mask else None
    if use_mask:
        mask[0] = 0                                      # attends nothing: the mean of its values
    cache, out, split, stream = kv.clone(), torch.empty(M, n_q, hd, device="cuda"), torch.empty(2, M, n_q, hd, dtype=torch.bfloat16, device="cuda"), torch.cuda.current_stream().cuda_stream
    size = lib().mn_attn_decode_workspace_bytes(M, n_q, hd, t_max)
    ws = torch.zeros(size // 4 + 64, dtype=torch.int32, device="cuda")
    ws[size // 4:] = 77
    arrived = dev.mn_attn_arrivals(M, n_q, n_kv, hd, t_max, ptr(ws), size, ctypes.byref(n))
    assert dev.mn_attn_decode_fused(ptr(qkv), qkv[0, 0].numel(), nz, qkv[0].numel(), M, n_q, n_kv, hd, 1, ptr(cos), ptr(sin), ptr(seq), ptr(slot), ptr(slot), 0, 0, hd ** -0.5, ptr(cache), t_max,
                                    ptr(length), ptr(mask), t_max if use_mask else 0, ptr(out), ptr(split), ptr(ws), arrived, stream) == 0
    x = qkv.double().sum(0)
    c, s = (t.double()[slot.long()][:, None] for t in (cos, sin))
    turn = lambda a: torch.cat([a[..., :half] * c - a[..., half:] * s, a[..., half:] * c + a[..., :half] * s], -1)  # noqa: E731
    q, k, v = turn(x[:, :n_q]) * hd ** -0.5, turn(x[:, n_q:n_q + n_kv]), x[:, n_q + n_kv:]
    want = torch.empty(M, n_q, hd, dtype=torch.float64, device="cuda")
    for m in range(M):
        at = int(slot[m])
        K, V = (kv[int(seq[m]), i, :, :at + 1].double() for i in (0, 1))
        K[:, at], V[:, at] = k[m], v[m]
        score = (K.repeat_interleave(n_q // n_kv, 0) @ q[m][:, :, None])[..., 0]
        if use_mask:
            score = score.masked_fill(mask[m, :at + 1] == 0, -torch.inf) if bool(mask[m, :at + 1].any()) else torch.zeros_like(score)
        want[m] = (torch.softmax(score, -1)[:, None] @ V.repeat_interleave(n_q // n_kv, 0))[:, 0]
        assert float((cache[int(seq[m]), 0, :, at].double() - k[m]).abs().max()) < 1e-5 and float((cache[int(seq[m]), 1, :, at].double() - v[m]).abs().max()) < 1e-5
    err = (out.double() - want).abs().amax((1, 2)) / want.abs().amax((1, 2))
    assert float(err.max()) < 3e-5, err
    assert float((split.double().sum(0) - out.double()).abs().max()) < 2.0 ** -16 * float(out.abs().max())
    assert bool((ws[size // 4:] == 77).all())
    if arrived:
        at = (arrived - ws.data_ptr()) // 4
        assert bool((ws[at:at + n.value] == 0).all())


@pytest.mark.parametrize("M", [64, 100, 200])
def test_a_long_row_is_shared(M):
    """Sixteen thousand keys of one row among short ones, walked by one workgroup a key head, took nine times as long as the step without them; a step of that row alone says what they cost."""
    def us(rows, longest):
        dec = decoder(8, 2, 128, 16384, rows)
        i32 = dict(dtype=torch.int32, device="cuda")
        x, seq, slot = torch.randn(rows, 256, device="cuda"), torch.arange(rows, **i32), torch.full((rows,), 100, **i32)
        slot[rows // 2] = longest
        length, out, best = slot + 1, torch.empty(rows, 256, device="cuda"), 1e9
        for _ in range(12):
            a, b = torch.cuda.Event(True), torch.cuda.Event(True)
            a.record()
            for _ in range(8):
                dec.step(x, seq, slot, slot, length, out=out, distinct_sequences=True)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best
    assert us(M, 16000) < us(M, 100) + 2 * us(1, 16000)


def test_replayed():
    """Captured with its counters: every replay starts and leaves them zero, with eager steps of the same workspace between."""
    M, t_max = 3, 700
    dec = decoder(8, 2, 128, t_max, M)
    g = torch.Generator().manual_seed(1)
    x, seq = torch.randn(M, 256, generator=g).cuda(), torch.arange(M, dtype=torch.int32).cuda()
    slot = torch.tensor([10, 300, 699], dtype=torch.int32).cuda()
    dec.kv_cache.normal_()
    length, out = slot + 1, torch.empty(M, 256, device="cuda")
    want = dec.step(x, seq, slot, slot, length, distinct_sequences=True).clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        dec.step(x, seq, slot, slot, length, out=out, distinct_sequences=True)
    torch.cuda.synchronize()
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(dec.step(x, seq, slot, slot, length, distinct_sequences=True), want)
        torch.cuda.synchronize()
