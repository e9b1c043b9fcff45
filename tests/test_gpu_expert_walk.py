"""Expert products of a decoder step, in the grid form or (many tiles) shared in equal parts by a resident set of workgroups, against the same rows one by one, which take neither: row
counts where the number of slabs changes, groups of one row and of all, blocks of 16 rows and one row more, layers on both sides of the rule.  bf16 hi / lo operands against fp32 ones,
two layers: 2^-17 each of a handful of products, 1e-4 of a row's norm.  And both forms by themselves against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def decoder(hidden, inter, experts, top, shared, n_seq):
    from ming_univision_amd import configuration as C
    from ming_univision_amd.bailing_moe import BailingMoeDecoder
    from ming_univision_amd.synth import synth_state_dict
    cfg = C.BailingMoeConfig(vocab_size=64, hidden_size=hidden, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2, num_experts=experts,
                             num_experts_per_tok=top, num_shared_experts=shared, moe_intermediate_size=inter, head_dim=128, use_bias=False,
                             image_patch_token=60, image_start_token=61)
    sd = {k: v.to("cuda", torch.bfloat16) for k, v in synth_state_dict(C.llm_param_shapes(cfg), 5, "cuda").items()}
    return BailingMoeDecoder.from_state_dict(cfg, sd, t_max=24, n_seq=n_seq)


@pytest.mark.parametrize("hidden,inter,experts,top,shared", [(1024, 1408, 64, 6, 2), (512, 200, 12, 12, 1), (256, 72, 4, 4, 2), (2048, 1408, 24, 3, 1)])
@pytest.mark.parametrize("rows", [3, 4, 5, 16, 17, 32, 33, 49, 64])
def test_rows_together_and_alone(rows, hidden, inter, experts, top, shared):
    from ming_univision_amd._lib import check, lib, ptr
    dec = decoder(hidden, inter, experts, top, shared, rows)
    g = torch.Generator(device="cuda").manual_seed(rows + hidden)
    x = torch.randn(rows, hidden, generator=g, device="cuda")
    past = torch.randn(dec.kv_cache.shape, generator=g, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    slot = i32([5 + r % 11 for r in range(rows)])

    def step(rs):
        routes = torch.full((2, len(rs), top + shared), -7, dtype=torch.int32, device="cuda")
        check(lib().mn_llm_route_capture(ptr(routes)), "mn_llm_route_capture")
        try:
            at = slot[rs].contiguous()
            out = dec.step(x[rs].contiguous(), i32(rs), at, at, at + 1, distinct_sequences=True).clone()
        finally:
            check(lib().mn_llm_route_capture(None), "mn_llm_route_capture")
        return out, routes.sort(dim=2).values
    dec.kv_cache.copy_(past)
    for ws in dec._ws.values():
        ws.fill_(127)                                    # what a slab does not hold is not read
    together, routes = step(list(range(rows)))
    dec.kv_cache.copy_(past)
    next(ws for (r, _), ws in dec._ws.items() if r == rows).fill_(255)        # (NaN everywhere)
    again, _ = step(list(range(rows)))
    assert torch.equal(together, again)
    dec.kv_cache.copy_(past)
    each = [step([r]) for r in range(rows)]
    alone, routes1 = torch.cat([o for o, _ in each]), torch.cat([r for _, r in each], dim=1)
    same = (routes == routes1).all(dim=2).all(dim=0)
    assert int((~same).sum()) <= (0 if experts == top else 1 + rows // 32)
    err = (together - alone).norm(dim=1) / alone.norm(dim=1)
    assert float(err[same].max()) < 1e-4, err


def internal(name):
    import ctypes
    import os
    from ming_univision_amd import _lib
    f = getattr(ctypes.CDLL(os.path.join(os.path.dirname(_lib.LIB_PATH), "libmingnative_dev.so")), name)
    f.restype, f.argtypes = _lib.SYMBOLS["mn_stream_mfma_grouped"]
    return f


def products(rows, G, slots, N, K):
    """A walk and a grid product of the same `slots` groups a row, as (slabs' sum, its float64 value, float64 sums of magnitudes)."""
    from ming_univision_amd import _lib
    from ming_univision_amd._lib import ptr
    walk = internal("mn_stream_kwalk_grouped")
    g = torch.Generator(device="cuda").manual_seed(rows + N + K)
    picks = torch.stack([torch.randperm(G, device="cuda", generator=g)[:slots] for _ in range(rows)]).flatten()
    order, count = torch.argsort(picks, stable=True), torch.bincount(picks, minlength=G)
    src = (order // slots).int().contiguous()
    off = torch.zeros(G + 1, dtype=torch.int32, device="cuda")
    off[1:] = count.cumsum(0)
    W = torch.empty(G, N, K, dtype=torch.bfloat16, device="cuda").normal_(0, K ** -0.5, generator=g)
    x = torch.randn(rows, K, device="cuda", generator=g)
    Y = torch.stack([x.bfloat16(), (x - x.bfloat16().float()).bfloat16()]).contiguous()
    x64, pairs = (Y[0].double() + Y[1].double())[src.long()], rows * slots
    parts = [(x64[int(off[e]):int(off[e + 1])], W[e].double().t()) for e in range(G)]
    want, size = torch.cat([a @ w for a, w in parts]), torch.cat([a.abs() @ w.abs() for a, w in parts])

    def run(f):
        out = torch.full((4 * pairs + 1, N), float("nan"), device="cuda")
        nz = f(ptr(Y), rows, ptr(W), N * K, ptr(out), pairs, ptr(off), ptr(src), G, rows, N, K, torch.cuda.current_stream().cuda_stream)
        assert 1 <= nz <= 4 and bool(out[nz * pairs:].isnan().all())
        return out[:nz * pairs].view(nz, pairs, N).sum(0).double()
    return run(walk), run(_lib.lib().mn_stream_mfma_grouped), want, size


@pytest.mark.parametrize("rows,N,K", [(16, 2816, 2048), (24, 2816, 2048), (24, 2048, 1408), (64, 2048, 1408)])
def test_error_of_whole_tiles(rows, N, K):
    """Enough tiles that a workgroup's share holds whole ones: their two chains of K / 2 are as long as those of the grid form's two ranges, so the error against float64 is that of the
    grid but for the draw; rounding errors grow with the square root of a chain's length or faster, so a single chain of K would be between 1.1 (where the operands' products are most of it) and 1.4 times as far."""
    walk, grid, want, _ = products(rows, 64, 8, N, K)
    walk, grid = (float((y - want).norm() / want.norm()) for y in (walk, grid))
    assert walk <= 1.05 * grid, (walk, grid)


@pytest.mark.parametrize("rows,G,slots,N,K", [(1, 1, 1, 1, 8), (3, 1, 1, 257, 64), (4, 4, 3, 72, 72), (5, 12, 12, 255, 128), (16, 8, 2, 384, 512), (17, 3, 3, 512, 200), (32, 256, 4, 40, 320),
                                              (33, 2, 2, 300, 1408), (64, 16, 1, 1024, 136), (64, 256, 16, 8, 64)])
def test_products(rows, G, slots, N, K):
    """Both forms at the edges: one group and 256, one row to 64 of a group, fewer chunks than workgroups, part chunks and part column tiles, one slab to four.  2 K products and their sums in fp32,
    in some order: 2^-24 of the magnitudes each."""
    walk, grid, want, size = products(rows, G, slots, N, K)
    bound = (2 * K + 16) * 2.0 ** -24 * size
    assert bool(((walk - want).abs() <= bound).all()) and bool(((grid - want).abs() <= bound).all())


@pytest.mark.parametrize("rows,G,slots,N,K,walks", [(16, 10, 4, 384, 512, 0), (5, 8, 4, 1408, 1024, 0), (5, 66, 6, 384, 256, 0), (3, 66, 8, 2816, 2048, 1), (24, 66, 8, 2048, 1408, 1)])
def test_few_tiles_take_the_grid(rows, G, slots, N, K, walks):
    """Two slabs are the grid's; the walk leaves three or four up to 32 rows.  Layers of few or small tiles took up to 1.7 times as long in the walk."""
    from ming_univision_amd._lib import ptr
    W, Y = torch.zeros(G, N, K, dtype=torch.bfloat16, device="cuda"), torch.zeros(2, rows, K, dtype=torch.bfloat16, device="cuda")
    pairs = rows * slots
    off = (torch.arange(G + 1, device="cuda") * pairs // G).to(torch.int32)
    src, out = torch.arange(pairs, device="cuda", dtype=torch.int32) % rows, torch.empty(4, pairs, N, device="cuda")
    f = internal("mn_stream_experts")
    f.argtypes = f.argtypes[:-1] + [f.argtypes[-2], f.argtypes[-1]]
    for two_slabs in (0, 1):                             # (and where the caller's scratch holds two: the grid whatever the tiles)
        nz = f(ptr(Y), rows, ptr(W), N * K, ptr(out), pairs, ptr(off), ptr(src), G, rows, N, K, two_slabs, torch.cuda.current_stream().cuda_stream)
        assert (nz > 2) == bool(walks and not two_slabs)


@pytest.mark.parametrize("rows,G,slots,N,K,walks", [(33, 48, 8, 1536, 2048, 0), (64, 48, 8, 1536, 2048, 0), (64, 17, 3, 4096, 2048, 0), (64, 66, 8, 2048, 1408, 1)])
def test_more_rows_take_the_grid(rows, G, slots, N, K, walks):
    """Above 32 rows a workgroup of the walk has a whole tile at least: fewer tiles than workgroups took a quarter longer than the grid, with experts that most rows like nearly twice as long.
    The walk zeros the second slab of a tile that one workgroup held; the grid has half of K there."""
    from ming_univision_amd._lib import ptr
    W, Y = torch.ones(G, N, K, dtype=torch.bfloat16, device="cuda"), torch.ones(2, rows, K, dtype=torch.bfloat16, device="cuda")
    pairs = rows * slots
    off = (torch.arange(G + 1, device="cuda") * pairs // G).to(torch.int32)
    src, out = torch.arange(pairs, device="cuda", dtype=torch.int32) % rows, torch.empty(2, pairs, N, device="cuda")
    f = internal("mn_stream_experts")
    f.argtypes = f.argtypes[:-1] + [f.argtypes[-2], f.argtypes[-1]]
    assert f(ptr(Y), rows, ptr(W), N * K, ptr(out), pairs, ptr(off), ptr(src), G, rows, N, K, 0, torch.cuda.current_stream().cuda_stream) == 2
    assert bool((out.sum(0) == 2 * K).all()) and bool((out[1] == 0).any()) == bool(walks)


@pytest.mark.parametrize("rows", [14, 15, 17])
def test_scratch_of_more_rows(rows):
    """Scratch sized for 65 rows holds a step of 14 .. 17 rows in two slabs a product, not in three: the step takes what there is.  Both orders of sums, fp32: 1e-4 of a row's norm as above."""
    import ctypes
    from ming_univision_amd._lib import lib
    dec = decoder(1024, 1408, 64, 6, 2, rows)
    g = torch.Generator(device="cuda").manual_seed(rows)
    x, i32 = torch.randn(rows, 1024, generator=g, device="cuda"), dict(dtype=torch.int32, device="cuda")
    seq, slot = torch.arange(rows, **i32), torch.full((rows,), 5, **i32)

    def step():
        dec.kv_cache.fill_(0.25)
        return dec.step(x, seq, slot, slot, slot + 1, distinct_sequences=True).clone()
    want = step()
    (key, full), n = next(iter(dec._ws.items())), lib().mn_llm_workspace_bytes(ctypes.byref(dec.struct), 65, dec.t_max)
    assert full.numel() > n
    buf = torch.full((n + 4096,), 77, dtype=torch.uint8, device="cuda")
    dec._ws[key] = buf[:n]
    got = step()
    assert bool((buf[n:] == 77).all())
    assert float(((got - want).norm(dim=1) / want.norm(dim=1)).max()) < 1e-4
