"""Decode graphs over latents that go by whole tiles a wave: the scratch taken once, for the longest sequence the cache holds, serves every shorter bound of the lengths."""
import pytest
import torch

from tests import pizitar_oracle as O
from tests.test_gpu_pizitar import err, run_portions, toks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rank,n_seq,length", [(512, 64, 1100), (256, 128, 1100), (384, 61, 1700)])
def test_graph_below_the_cache_length(rank, n_seq, length):
    """64 sequences over latents of 512: 16 splits at 2048 tokens, 20 at 1280.  Every sequence holds the same tokens, every row of every replay against the float64 oracle (1e-4 of the
    logits' scale, as the other decoding tests)."""
    from ming_univision_amd.configuration import PizitarConfig
    from ming_univision_amd.pizitar import PizitarDecoder
    cfg = O.random_config([dict(type="latent_attention", heads=2, dim=16, vdim=16, kv_rank=rank, q_rank=16, ff=32)], width=32, vocab=40, taps=2)
    sd = O.random_weights(cfg, 3, 1.0)
    dec = PizitarDecoder(PizitarConfig.from_dict(cfg), {k: v.cuda() for k, v in sd.items()}, t_max=2048, n_seq=n_seq, arith="f32")
    t = toks(cfg, length + 4, 5)
    ref = O.logits_of(cfg, sd, t)
    run_portions(dec, 0, t[:length], [length])
    for a in dec.latent:
        a[1:] = a[:1]
    dec.taps_state[:, 1:] = dec.taps_state[:, :1]
    row_seq = torch.arange(n_seq, dtype=torch.int32, device="cuda")
    slot = torch.full((n_seq,), length, dtype=torch.int32, device="cuda")
    g = dec.decode_graph(row_seq, slot, slot + 1)
    for i in range(4):
        hid = g.run(dec.embed(torch.full((n_seq,), t[length + i], device="cuda")), length + i + 1)
        lg = dec.logits(hid.clone())
        torch.cuda.synchronize()
        assert g.bound < dec.t_max and err(lg, ref[length + i][None].expand(n_seq, -1)) < 1e-4, i


def test_fewer_splits_than_the_scratch_holds():
    """mn_latent_attn where the caller's splits are more than one round of workgroups (64 rows over 1280 keys in 20): the result is a split's result, and nothing beyond the scratch is written."""
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    g = torch.Generator().manual_seed(9)
    M, H, r, t_max, ks = 64, 16, 512, 1280, 20
    q, arena = (torch.randn(M, H, r, generator=g) * 2 * r ** -0.5).cuda(), torch.randn(4, t_max, r, generator=g).cuda()
    seq, lens = torch.arange(M, dtype=torch.int32, device="cuda") % 4, torch.full((M,), t_max, dtype=torch.int32, device="cuda") - torch.arange(M, dtype=torch.int32, device="cuda")
    blk = torch.stack([torch.arange(M, dtype=torch.int32), torch.ones(M, dtype=torch.int32)], 1).cuda()
    n = lib().mn_latent_attn_workspace_bytes(M, H, r, ks)
    ws, out = torch.full((n + 4096,), 77, dtype=torch.uint8, device="cuda"), torch.empty(M, H, r, device="cuda")
    check(lib().mn_latent_attn(ptr(q), ptr(arena), ptr(seq), ptr(lens), ptr(blk), M, M, H, r, t_max, t_max, ks, ptr(out), ptr(ws), n, current_stream()), "latent")
    assert bool((ws[n:] == 77).all())
    for m in range(0, M, 7):
        k = arena[seq[m], :lens[m]].double()
        want = torch.softmax(q[m].double() @ k.T, -1) @ k
        assert float((out[m] - want).norm() / want.norm()) < 1e-6


@pytest.mark.parametrize("r,n,length", [(512, 5, 160), (512, 4, 320), (384, 9, 96), (256, 5, 128), (256, 4, 160)])
def test_prompts_on_both_sides_of_the_line(r, n, length):
    """Prompts of n sequences, 16 heads: more workgroups than rounds of them are worth whole tiles a wave, and on the other side of that line."""
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    g = torch.Generator().manual_seed(r + n)
    M, H = n * length, 16
    q, arena = (torch.randn(M, H, r, generator=g) * 2 * r ** -0.5).cuda(), torch.randn(n, length, r, generator=g).cuda()
    seq, lens = torch.arange(M, dtype=torch.int32, device="cuda") // length, torch.arange(M, dtype=torch.int32, device="cuda") % length + 1
    blk = torch.stack([torch.arange(0, M, 4, dtype=torch.int32), torch.full((M // 4,), 4, dtype=torch.int32)], 1).cuda()
    ks = lib().mn_latent_attn_splits(M // 4 * 4, length, r)
    ws, out = torch.empty(max(16, lib().mn_latent_attn_workspace_bytes(M, H, r, ks)), dtype=torch.uint8, device="cuda"), torch.empty(M, H, r, device="cuda")
    check(lib().mn_latent_attn(ptr(q), ptr(arena), ptr(seq), ptr(lens), ptr(blk), M // 4, M, H, r, length, length, ks, ptr(out), ptr(ws), ws.numel(), current_stream()), "latent")
    for i in range(n):
        rows = slice(i * length, (i + 1) * length)
        k = arena[i].double()
        see = torch.arange(length, device="cuda")[None] <= torch.arange(length, device="cuda")[:, None]
        s = (q[rows].double() @ k.T).masked_fill(~see[:, None], -float("inf"))
        want = torch.softmax(s, -1) @ k
        assert float((out[rows] - want).norm() / want.norm()) < 1e-6
