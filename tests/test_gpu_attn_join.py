"""Decode attention that appends the new key itself and splits a row's keys over workgroups, the last of which joins them (decoder steps of rows of distinct sequences), against
the launches that steps without that promise take: rows of one key, at the edges of a batch of keys and of the first split, up to the cache's end; row counts from one row to more than
a workgroup a CU; one to four query heads a key head of 64 and of 128; holes in the mask and a row that attends nothing; one long row among short ones (splits by the rows' lengths up to 128
rows, of 1024 keys above).  Both sum fp32 products of at most 9000 keys in
another order (1e-6 of the largest value), two layers and the products between them pass it on: 2e-5 of a row's norm."""
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
